// Part of htr_gfx950.hip, included inside its anonymous namespace: k_linear_tile: 17 to 64 activation rows, and grouped launches of more than 8.
// ------------------------------------------------------------------------------------------------ tiles of 32 JB rows
// A workgroup owns one 128-row block of the weight, up to 32 JB activation rows and 1/S of the column blocks.  Wave w =
// (row half rh = w % 2, column quarter cq = w / 2) decodes 64 weight rows x 32 columns per 128-column step, one granule
// (two rows x 16 columns of a tile) per lane: lane = (tile column 2 cq + lane / 32, strip 4 rh + lane % 32 / 8, row pair
// lane % 8).  The decode registers are the A operands of v_mfma_f32_32x32x16_f16 as they are: the k-slots of lanes 0..31
// stand for columns of tile column 2 cq, those of lanes 32..63 for tile column 2 cq + 1, first columns 0..7 of both, then
// columns 8..15, for the even and for the odd row of the pair: four operands, 32 weight rows each.
// The B operands come straight from memory: the rotation ahead of the launch leaves the activations in the order in which
// the lanes want them (fragments of 32 rows x 16 columns, 1 KB each), so a wave reads its own fragments with fully
// coalesced loads, ahead of their use, and there is neither staging through LDS nor a barrier in the loop: the waves run
// freely, and one wave's matrix instructions overlap the others' decode.
// Bound: vector issue of the decode (K4: 873 cycles per step and SIMD of two waves; measured 0.40 us per step with one tile
// of 32 rows, 0.53 with two, where k_linear_batch with its staging and barrier takes 0.49 and 0.69), then 6.7 to 8.6 us per
// launch for launch, first loads, reduction and output side.  32x32x16 instead of 16x16x32 instructions because one of
// them takes about 6 cycles of vector issue from the other waves for 16 K products, and the smaller one 12 for 8 K.
// ONE (a single column split: tall matrices, groups that fill the chip, routed experts): two workgroups per compute unit.  A
// workgroup of 16 steps spends as long on its first loads and its output side as on a third of its steps; 500 tokens over 64
// experts, 47 rows each on average, two row tiles: gate/up 130 -> 95 us, down 80 -> 57 us.
constexpr int FLAG_ENTRY_TILES = 1 << 6;                                    // grouped: an entry's `reserved` is its first row tile
constexpr int TILE_FIN_LD = 128 + 4;                                        // floats per activation row of the output in LDS
constexpr size_t tile_lds_bytes(int jb) { return (size_t)2 * 32 * jb * TILE_FIN_LD * 4 + 2 * 32 * jb * 4; }

template <int K, int JB, int P, int DB, bool ONE>
__global__ __launch_bounds__(WG_THREADS, ONE ? 4 : 2) void k_linear_tile(const uint32_t* __restrict__ qw_a, float* __restrict__ part,
                                                                         int m, int n, int M_a, int S_a, int flags, const LinearTail t_a) {
  extern __shared__ __align__(16) unsigned char lds[];
  const uint32_t* __restrict__ qw = qw_a;
  LinearTail t = t_a;
  int M = M_a;
  const int S = ONE ? 1 : S_a;
  if (t_a.group != nullptr) {                      // uniform: one entry of the problem table per blockIdx.z
    const htr_group_entry& ge = t_a.group[blockIdx.z];
    M = ge.M;
    if (M <= 0) return;
    qw = (const uint32_t*)ge.qweight;
    t.scales = (const uint16_t*)ge.scales; t.sv = (const uint8_t*)ge.sv; t.bias = ge.bias; t.y = ge.y;
    // first row tile of the problem: given (routed experts), or one tile per problem
    const size_t tile0 = (flags & FLAG_ENTRY_TILES) ? (size_t)ge.reserved : (size_t)blockIdx.z;
    t.xt_g = t_a.xt_g + tile0 * 32 * n;
    t.xs_g = t_a.xs_g + tile0 * 32 * (n >> 7) * 4;
    t.sc_g = t_a.sc_g + tile0 * 32;
    if (!ONE) part += (size_t)blockIdx.z * gridDim.y * S * M_a * 128;      // M_a: the largest M of the group
  }
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int rh = w & 1, cq = w >> 1, l32 = lane & 31, kg = lane >> 5;
  const int nblk = n >> 7;
  const int s_idx = blockIdx.x, rb = blockIdx.y;
  const int cb = (nblk + S - 1) / S;
  const int c_begin = s_idx * cb, c_end = min(nblk, c_begin + cb);
  const int nsteps = c_end - c_begin;              // >= 1: the host picks S so that no split is empty
  const int y_dtype = (flags >> 2) & 3;
  constexpr int ROWS = 32 * JB;
  float* s_fin = (float*)lds;                      // [2][ROWS][TILE_FIN_LD]
  float* s_off = s_fin + 2 * ROWS * TILE_FIN_LD;   // [ROWS] 1534 x sum of the rotated activations over the split
  float* s_sc = s_off + ROWS;                      // [ROWS] activation scale
  constexpr uint32_t OUT_OF_RANGE = 0x7FFFF000u;     // beyond every descriptor, with all the steps that are added to it

  // ---- requests: the first fragments and weights
  const int jbs = (M + 31) >> 5;                   // row tiles that hold rows
  const __amdgpu_buffer_rsrc_t brsrc = __builtin_amdgcn_make_buffer_rsrc((void*)t.xt_g, 0, jbs * 32 * n * 2, 0x00020000);
  uint32_t boff[JB];
#pragma unroll
  for (int jb = 0; jb < JB; ++jb) boff[jb] = 32 * jb + l32 < M ? (uint32_t)((jb * (n >> 5) + c_begin * 4 + cq) * 2048 + lane * 16) : OUT_OF_RANGE;
  h8 B[DB][JB][2];
  int b_left = nsteps;
  auto load_b = [&](int set) {                     // fragments of the next step not yet requested
    HTR_PIN();
#pragma unroll
    for (int jb = 0; jb < JB; ++jb) {
      const uint32_t o = b_left > 0 ? boff[jb] : OUT_OF_RANGE;          // rows beyond M, steps beyond the split: zeros, no traffic
      B[set][jb][0] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(brsrc, o, 0, 0));
      B[set][jb][1] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(brsrc, o + 1024, 0, 0));
      boff[jb] += 4 * 2048;
    }
    --b_left;
    HTR_PIN();
  };
  const SplitRole role = ONE ? SplitRole{1, 0, false, true} : split_role(M, S, s_idx, flags);
  RowBits raw = {0u, 0u, 0u, 0u, 0u, 0u};
  if (role.finisher) load_row_bits(t, y_dtype, rb * 128 + lane, raw);
  constexpr int STEP_BYTES = 256 * K;
  const uint32_t strip_bytes = (uint32_t)nblk * STEP_BYTES;
  const uint32_t* base = qw + ((size_t)(rb * 8) * nblk + (size_t)c_begin) * (STEP_BYTES / 4);
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)(7u * strip_bytes + (uint32_t)nsteps * STEP_BYTES), 0x00020000);
  uint32_t pf_off = (4 * rh + (l32 >> 3)) * strip_bytes + ((2 * cq + kg) * 8 + (lane & 7)) * 4 * K;
  int pf_left = nsteps;
  StreamRegs<K> buf[P];
  auto prefetch = [&](StreamRegs<K>& dst) {
    HTR_PIN();
    load_stream_buffer<K>(rsrc, pf_left > 0 ? pf_off : OUT_OF_RANGE, dst);
    pf_off += STEP_BYTES;
    --pf_left;
    HTR_PIN();
  };
#pragma unroll
  for (int p = 0; p < DB; ++p) { if (p < P) prefetch(buf[p]); load_b(p); }
#pragma unroll
  for (int p = DB; p < P; ++p) prefetch(buf[p]);

  // sums of the rotated activations over the split's columns: 512 / ROWS (a power of two) lanes per row
  {
    constexpr int LPR = WG_THREADS / ROWS;
    const int row = (int)threadIdx.x / LPR, sub = (int)threadIdx.x % LPR;
    float v = 0.f;
    if (row < M)
      for (int b = c_begin + sub; b < c_end; b += LPR) {
        const f2 q = *(const HTR_GLOBAL f2*)((const HTR_GLOBAL float*)t.xs_g + ((size_t)row * nblk + b) * 4);
        v += q.x + q.y;
      }
    v += dpp_mov<0xB1>(v); v += dpp_mov<0x4E>(v);
    if constexpr (LPR >= 8) v += dpp_mov<0x141>(v);
    if constexpr (LPR >= 16) v += dpp_mov<0x140>(v);
    if (sub == 0 && row < ROWS) {
      s_off[row] = 1534.f * v;
      s_sc[row] = row < M ? ((const HTR_GLOBAL float*)t.sc_g)[row] : 0.f;
    }
  }

  f16v acc[JB][2];
#pragma unroll
  for (int jb = 0; jb < JB; ++jb)
#pragma unroll
    for (int par = 0; par < 2; ++par)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[jb][par][r] = 0.f;
  const int hist = history_lane_byteaddr(lane);
  auto multiply = [&](const DecodedStep<K>& d, int set) {      // d.a[0], d.a[1] = even row columns 0..7, 8..15; d.a[2], d.a[3] = odd row
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int jb = 0; jb < JB; ++jb) {
        acc[jb][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(d.a[hf], B[set][jb][hf], acc[jb][0], 0, 0, 0);
        acc[jb][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(d.a[2 + hf], B[set][jb][hf], acc[jb][1], 0, 0, 0);
      }
  };
  static_assert(P % DB == 0 || DB % P == 0, "both rings rotate with the unrolled loop");
  constexpr int U = P > DB ? P : DB;
  DecodedStep<K> cur;
  decode_step<K>(buf[0], hist, cur);
  prefetch(buf[0]);
  int v = 0;
  for (; v + U < nsteps; v += U) {
#pragma unroll
    for (int pp = 0; pp < U; ++pp) {
      multiply(cur, pp % DB);
      load_b(pp % DB);
      decode_step<K>(buf[(pp + 1) % P], hist, cur);
      prefetch(buf[(pp + 1) % P]);
    }
  }
#pragma unroll
  for (int pp = 0; pp < U; ++pp) {
    if (v + pp < nsteps) {
      multiply(cur, pp % DB);
      if (v + pp + 1 < nsteps) {
        load_b(pp % DB);
        decode_step<K>(buf[(pp + 1) % P], hist, cur);
        prefetch(buf[(pp + 1) % P]);
      }
    }
  }

  // ---- the four column quarters meet in LDS, in two copies: D[i][j]: lane holds column j = lane % 32 (activation row), register
  // r row i = 8 (r / 4) + 4 kg + r % 4; row i of an A operand is strip 4 rh + i / 8, row pair i % 8, so a lane's values for
  // r = 4 rq .. 4 rq + 3, both parities interleaved, are the 8 consecutive weight rows 64 rh + 16 rq + 8 kg ..
  __syncthreads();                                  // s_off, s_sc
  float scl[JB], off[JB];
#pragma unroll
  for (int jb = 0; jb < JB; ++jb) { scl[jb] = s_sc[32 * jb + l32]; off[jb] = cq == 0 ? s_off[32 * jb + l32] : 0.f; }
#pragma unroll
  for (int phase = 0; phase < 2; ++phase) {
    if ((cq >> 1) == phase) {
      float* copy = s_fin + (cq & 1) * (ROWS * TILE_FIN_LD);
#pragma unroll
      for (int jb = 0; jb < JB; ++jb) {
        float* dst = copy + (32 * jb + l32) * TILE_FIN_LD + 64 * rh + 8 * kg;
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          f4 lo = {(acc[jb][0][4 * rq] - off[jb]) * scl[jb], (acc[jb][1][4 * rq] - off[jb]) * scl[jb],
                   (acc[jb][0][4 * rq + 1] - off[jb]) * scl[jb], (acc[jb][1][4 * rq + 1] - off[jb]) * scl[jb]};
          f4 hi = {(acc[jb][0][4 * rq + 2] - off[jb]) * scl[jb], (acc[jb][1][4 * rq + 2] - off[jb]) * scl[jb],
                   (acc[jb][0][4 * rq + 3] - off[jb]) * scl[jb], (acc[jb][1][4 * rq + 3] - off[jb]) * scl[jb]};
          if (phase == 1) { lo += *(const f4*)(dst + 16 * rq); hi += *(const f4*)(dst + 16 * rq + 4); }
          *(f4*)(dst + 16 * rq) = lo;
          *(f4*)(dst + 16 * rq + 4) = hi;
        }
      }
    }
    __syncthreads();
  }
  finish_row_block<JB * 4>(t, part, rb, m, M, role, raw, s_fin, TILE_FIN_LD, ROWS * TILE_FIN_LD, lane, lane + 64, w, lane, y_dtype);
}
