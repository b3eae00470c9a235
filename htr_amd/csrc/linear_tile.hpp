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

// ---- output side of a row block for tiles.  What finish_row_block does (same slots, same owners of the activation rows), with
// four activation rows to a wave, 16 lanes each: lane i holds output rows i, 16 + i, .. 112 + i, so bits 4 to 6 of H128 are
// additions between its registers; through the row's place in LDS it gets rows 8 i .. 8 i + 7, so bits 0 to 2 are again, bit 3 is
// a DPP exchange, and the eight results leave in one or two 16-byte stores.  About 28 vector instructions per activation row where
// one row to a wave, two output rows to a lane, takes 75: there every butterfly stage is an exchange.  Bound: latency of the LDS
// trips, then vector issue.  500 tokens over 64 experts (2048x1408, K4, two row tiles): gate/up 98 -> 93 us, down 58 -> 54.
// Row constants come through LDS: 64 groups of four words (scales in the order in which a lane takes them, then biases) and 16
// sign bytes, a word each.
struct RowConsts { float* groups; int stride; uint32_t* signs; };           // stride: floats from one group to the next
__device__ __forceinline__ void place_row_consts(const LinearTail& t, const RowBits& raw, int y_dtype, int lane, const RowConsts& c) {
  auto cvt_bias = [&](uint32_t b) {
    return y_dtype == HTR_F32 ? __uint_as_float(b) : y_dtype == HTR_BF16 ? bf16_bits_to_float((uint16_t)b) : f16_bits_to_float((uint16_t)b);
  };
  float* rs = c.groups + (lane & 15) * 2 * c.stride + (lane >> 4);          // output row 16 j + i is word 8 i + j
  rs[0] = f16_bits_to_float((uint16_t)raw.sc0) * t.cbscale * INV_SQRT128;
  rs[c.stride] = f16_bits_to_float((uint16_t)raw.sc1) * t.cbscale * INV_SQRT128;
  float* bs = c.groups + (32 + (lane >> 2)) * c.stride + (lane & 3);
  bs[0] = cvt_bias(raw.b0);
  bs[16 * c.stride] = cvt_bias(raw.b1);
}
__device__ __forceinline__ void place_row_signs(const RowBits& raw, int lane, const RowConsts& c) {
  if ((lane & 7) == 0) { c.signs[lane >> 3] = raw.sv0; c.signs[8 + (lane >> 3)] = raw.sv1; }
}
__device__ __forceinline__ void butterflies8(float (&v)[8]) {               // H8 over the index
#pragma unroll
  for (int h = 1; h < 8; h <<= 1)
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (!(k & h)) { const float a = v[k], b = v[k | h]; v[k] = a + b; v[k | h] = a - b; }
}
// eight consecutive values of an output row; 16-byte stores where the output starts on such a boundary
__device__ __forceinline__ void store8(void* y, int y_dtype, size_t idx, const float (&v)[8]) {
  if (((uintptr_t)y & 15) == 0) {
    if (y_dtype == HTR_F32) {
      HTR_GLOBAL f4* p = (HTR_GLOBAL f4*)((HTR_GLOBAL float*)y + idx);
      p[0] = f4{v[0], v[1], v[2], v[3]};
      p[1] = f4{v[4], v[5], v[6], v[7]};
    } else {
      typedef float f8 __attribute__((ext_vector_type(8)));
      const f8 q = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
      *(HTR_GLOBAL u4*)((HTR_GLOBAL uint16_t*)y + idx) =
          y_dtype == HTR_BF16 ? __builtin_bit_cast(u4, __builtin_convertvector(q, b8)) : __builtin_bit_cast(u4, __builtin_convertvector(q, h8));
    }
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k) store_elem_g(y, y_dtype, idx + k, v[k]);
  }
}
// s_fin: [activation row][TILE_FIN_LD], with TWO two copies to be added, the second `copy` floats behind the first.  ONE: a single split.
template <bool ONE, bool TWO>
__device__ __forceinline__ void finish_tile(const LinearTail& t, void* y, float* __restrict__ part, int rb, int m, int M, const SplitRole& role,
                                            float* s_fin, int copy, const RowConsts& consts, uint32_t stale, int w, int lane, int y_dtype) {
  const int S = ONE ? 1 : role.S, s_idx = ONE ? 0 : role.s_idx, RG = (M + 7) >> 3;
  const bool spread = ONE ? false : role.spread;
  if (!ONE) {
    for (int rg = 0, owner = spread ? 0 : S - 1; rg < RG; ++rg, owner = !spread ? owner : (owner + 1 == S ? 0 : owner + 1)) {
      const int mrow = 8 * rg + w;
      if (owner != s_idx && mrow < M) {
        const float* own = s_fin + mrow * TILE_FIN_LD;
        const float* oth = own + copy;
        uint32_t* dst = (uint32_t*)(part + (((size_t)rb * S + s_idx) * M + mrow) * 128);
        __hip_atomic_store(dst + lane, __float_as_uint(TWO ? own[lane] + oth[lane] : own[lane]) | 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(dst + lane + 64, __float_as_uint(TWO ? own[lane + 64] + oth[lane + 64] : own[lane + 64]) | 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (!role.finisher) return;
  }
  const int i = lane & 15;
  float rs[8], bias[8];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const f4 r = *(const f4*)(consts.groups + (2 * i + h) * consts.stride), b = *(const f4*)(consts.groups + (32 + 2 * i + h) * consts.stride);
    rs[4 * h] = r.x; rs[4 * h + 1] = r.y; rs[4 * h + 2] = r.z; rs[4 * h + 3] = r.w;
    bias[4 * h] = b.x; bias[4 * h + 1] = b.y; bias[4 * h + 2] = b.z; bias[4 * h + 3] = b.w;
  }
  const uint32_t signs = consts.signs[i];
  const float s1 = (i & 1) ? -1.f : 1.f;
  // the o-th activation row that this split finishes; a wave takes rows o, o + 4, o + 8, o + 12 at once, whose places in LDS
  // are 16 banks apart
  const int mine = 8 * (spread ? (RG - s_idx + S - 1) / S : RG), o0 = 16 * (w >> 2) + (w & 3) + 4 * (lane >> 4);
  auto row_of = [&](int o) { return o < mine ? 8 * (spread ? s_idx + (o >> 3) * S : o >> 3) + (o & 7) : M; };
  // slot of the k-th other split for an activation row
  auto slot_of = [&](int k, int mrow) { return (uint32_t*)(part + (((size_t)rb * S + k + (k >= s_idx ? 1 : 0)) * M + mrow) * 128) + i; };
  // the output side of one row; v = the other splits' sum
  auto finish_row = [&](int mrow, float (&v)[8], bool failed) {
    float* own = s_fin + mrow * TILE_FIN_LD;
    const float* oth = own + copy;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (v[j] + (TWO ? own[16 * j + i] + oth[16 * j + i] : own[16 * j + i])) * rs[j];
    butterflies8(v);
#pragma unroll
    for (int j = 0; j < 8; ++j) own[16 * j + i] = v[j];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");                    // the row's 16 lanes are in one wave
    __builtin_amdgcn_wave_barrier();
    const f4 lo = *(const f4*)(own + 8 * i), hi = *(const f4*)(own + 8 * i + 4);
    v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
    butterflies8(v);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      butterfly_dpp<1>(v[k], s1);
      v[k] = __uint_as_float(__float_as_uint(v[k]) ^ ((signs << (31 - k)) & 0x80000000u)) + bias[k];
      if (failed) v[k] = __builtin_nanf("");
    }
    store8(y, y_dtype, (size_t)mrow * m + rb * 128 + 8 * i, v);
  };
  if (ONE || S == 1) {
    for (int o = o0; row_of(o) < M; o += 32) {
      float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      finish_row(row_of(o), v, stale != 0u);
    }
    return;
  }
  // With other splits: the slots of up to RB of the wave's rows (JW splits each) are requested together, so that the rows behind
  // the first cost no memory round trip of their own; repeated (bounded) until every partial is there, summed in fixed order.
  auto finish_rows = [&](auto jw_c, auto rb_c) {
    constexpr int JW = decltype(jw_c)::value, RB = decltype(rb_c)::value;
    for (int o = o0; row_of(o) < M; o += 32 * RB) {
      float sum[RB][8];
      bool failed = false;
      int tries = 0;
      for (;;) {
        uint32_t u[RB][JW][8];
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const int mrow = row_of(o + 32 * r) < M ? row_of(o + 32 * r) : row_of(o);       // beyond the last row: the first again, not looked at
#pragma unroll
          for (int k = 0; k < JW; ++k) {
            const uint32_t* pp = slot_of(min(k, S - 2), mrow);
#pragma unroll
            for (int j = 0; j < 8; ++j) u[r][k][j] = __hip_atomic_load(pp + 16 * j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
        bool missing = false;
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const bool real = row_of(o + 32 * r) < M;
#pragma unroll
          for (int j = 0; j < 8; ++j) sum[r][j] = 0.f;
#pragma unroll
          for (int k = 0; k < JW; ++k)
            if (real && k < S - 1)
#pragma unroll
              for (int j = 0; j < 8; ++j) { missing |= u[r][k][j] == 0u; sum[r][j] += __uint_as_float(u[r][k][j]); }
        }
        if (!__any(missing)) break;
        if (++tries >= t.spin_limit) { failed = true; break; }
        __builtin_amdgcn_s_sleep(2);
      }
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const int mrow = row_of(o + 32 * r);
        if (mrow >= M) continue;
        if (!failed) {                                                        // slots back to zero for the next call
          for (int k = 0; k < S - 1; ++k) {
            uint32_t* pp = slot_of(k, mrow);
#pragma unroll
            for (int j = 0; j < 8; ++j) __hip_atomic_store(pp + 16 * j, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        } else if (i == 0) {
          report_give_up(t.status);
        }
        finish_row(mrow, sum[r], failed || stale != 0u);
      }
    }
  };
  if (S == 2) finish_rows(std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{});
  else if (S <= 4) finish_rows(std::integral_constant<int, 3>{}, std::integral_constant<int, 2>{});
  else finish_rows(std::integral_constant<int, 7>{}, std::integral_constant<int, 1>{});
}
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
  // row constants of the output side: in the four floats behind each of the 64 JB rows, signs later in the place of s_off
  const RowConsts consts = {s_fin + 128, TILE_FIN_LD, (uint32_t*)s_off};
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
  // ONE, one row tile: few rows of many experts.  Up to 8 rows a wave finishes one row by itself, with no trip through LDS: half a
  // microsecond of the 45 us that both products of 16 tokens over 64 experts take.
  constexpr bool FEW = ONE && JB == 1;
  const bool few = FEW && M <= 8;
  if (role.finisher && (w == 0 || few)) load_row_bits(t, y_dtype, rb * 128 + lane, raw);
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
  if (role.finisher && w == 0 && !few) place_row_consts(t, raw, y_dtype, lane, consts);
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
    if (phase == 1 && role.finisher && w == 0 && !few) place_row_signs(raw, lane, consts);      // every wave has its offsets
    __syncthreads();
  }
  if constexpr (FEW) {
    if (few) {
      finish_row_block<1>(t, part, rb, m, M, role, raw, s_fin, TILE_FIN_LD, ROWS * TILE_FIN_LD, lane, lane + 64, w, lane, y_dtype);
      return;
    }
  }
  const uint32_t stale = t.status != nullptr ? load_status(t.status) : 0u;     // non-zero: an earlier launch on this workspace gave up
  finish_tile<ONE, true>(t, t.y, part, rb, m, M, role, s_fin, ROWS * TILE_FIN_LD, consts, stale, w, lane, y_dtype);
}
