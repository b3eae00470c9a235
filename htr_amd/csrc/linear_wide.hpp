// Part of htr_gfx950.hip, included inside its anonymous namespace: k_linear_wide: many activation rows, the weight decoded once per
// 256 of them.
// ------------------------------------------------------------------------------------------------ wide tiles
// A workgroup owns one 128-row block of the weight, one tile of 256 activation rows and 1/S of the column blocks; the last tile,
// which may hold fewer rows and then takes less time per column block, has a split of its own (grid = tiles x row blocks x splits).  What a wave decodes goes through LDS and serves all activation rows of the tile, where k_linear_gemm's
// waves keep what they decode for themselves and repeat the decode for every 96 or 128 rows.
//   decode  = wave w = (row half rh = w % 2, column quarter cq = w / 2) of every 128-column block, lane = (tile column 2 cq + lane / 32,
//             strip 4 rh + lane % 32 / 8, row pair lane % 8) as in k_linear_tile, one block ahead of the products.
//   A       = fragments (32-column unit u, half hf, 32-row piece b) of 1 KB, lane (kg = lane / 32, i = lane % 32) of a matrix
//             instruction at 16 lane: tile column kg of the unit, columns 8 hf .. + 7, row i of piece b = strips 2b, 2b + 1, i = 16 x
//             row parity + 8 x strip parity + row pair: a decoding lane writes its granule as four 16-byte pieces, 16 lanes side
//             by side.  Two buffers of 32 KB, one barrier per block.
//   B       = the rotated activations in the fragment order of linear.hpp.  Wave w multiplies the 32 activation rows 32 w .. of the
//             tile with all 128 weight rows, so no other wave needs its fragments and they go from memory to its registers, two
//             blocks ahead.  (Through LDS they would cost more of it than it has: it reads 256 bytes a cycle but writes 78.)
//   product = per block 32 v_mfma_f32_32x32x16_f16 with a 16-byte LDS read each, three to four vector instructions of the decode
//             between two of them.
// The decoded halves are centred (v instead of 1534 + v, exact; a packed subtraction for two weights, in the shadow of the matrix
// instructions), so no sums of the activations are needed for an offset, which the first block would wait for.
// The accumulators are complete sums over the split, so the output side needs no reduction over the waves (finish_tile).
constexpr int WIDE_ROWS = 256;
constexpr int WIDE_A = 32768;                                   // bytes of a block's A fragments
constexpr size_t WIDE_SMALL = (size_t)WIDE_ROWS * TILE_FIN_LD * 4;        // [rows] scales, row constants (272 words) behind the output
constexpr size_t WIDE_LDS = WIDE_SMALL + (size_t)(WIDE_ROWS + 272) * 4;
static_assert(WIDE_SMALL >= 2 * WIDE_A, "the output takes the place of the operands");

__device__ __forceinline__ uint32_t centred(uint32_t pair) {     // two halves 1534 + v -> v
  const h2 c = {(_Float16)-1534.f, (_Float16)-1534.f};
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, pair) + c);
}

template <int K>
__global__ __launch_bounds__(WG_THREADS) void k_linear_wide(const uint32_t* __restrict__ qw, float* __restrict__ part, int m, int n, int M_all,
                                                            int S_full, int S_last, int flags, const LinearTail t) {
  extern __shared__ __align__(16) unsigned char lds[];
  constexpr int ROWS = WIDE_ROWS, P = 2;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rh = w & 1, cq = w >> 1, l32 = lane & 31, kg = lane >> 5;
  const int nblk = n >> 7;
  // splits of a row block are consecutive workgroups
  const int id = blockIdx.x, rbs = m >> 7, last = (M_all - 1) / ROWS, id_last = last * rbs * S_full;
  const bool is_last = id >= id_last;
  const int S = is_last ? S_last : S_full, mt = is_last ? last : id / (rbs * S_full), id0 = is_last ? id_last : mt * rbs * S_full;
  const int rb = (id - id0) / S, s_idx = id - id0 - rb * S;
  const int j0 = mt * ROWS, M = min(ROWS, M_all - j0);           // this tile's activation rows
  const int cb = (nblk + S - 1) / S;
  const int c_begin = s_idx * cb, c_end = min(nblk, c_begin + cb);
  const int nsteps = c_end - c_begin;                            // >= 1: the host picks S so that no split is empty
  const int y_dtype = (flags >> 2) & 3;
  float* s_fin = (float*)lds;                                    // [ROWS][TILE_FIN_LD], over the operands once the products are done
  float* s_sc = (float*)(lds + WIDE_SMALL);                      // [ROWS] activation scale
  const RowConsts consts = {s_sc + ROWS, 4, (uint32_t*)(s_sc + ROWS + 256)};
  constexpr uint32_t OUT_OF_RANGE = 0x7FFFF000u;

  // ---- this wave's activations; rows beyond M read the tile's last row: their products are not looked at
  const bool active = 32 * w < M;                                // uniform
  const __amdgpu_buffer_rsrc_t brsrc = __builtin_amdgcn_make_buffer_rsrc((void*)t.xt_g, 0, M_all * n * 2, 0x00020000);
  const int jt = min((j0 >> 5) + w, (M_all - 1) >> 5), tr = min(32, M_all - 32 * jt);
  const uint32_t frag_bytes = 32u * (uint32_t)tr;
  const uint32_t boff = (uint32_t)jt * 64u * (uint32_t)n + (uint32_t)(kg * tr + min(l32, tr - 1)) * 16u;
  h8 B[2][8];
  auto load_b = [&](int set, int uf, int step) {                 // step within the split; beyond its last: that one again
    const uint32_t so = (uint32_t)((c_begin + min(step, nsteps - 1)) * 8 + uf) * frag_bytes;
    B[set][uf] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(brsrc, boff, so, 0));
  };
  // ---- the weight stream
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
  const SplitRole role = split_role(M, S, s_idx, flags);
  RowBits raw = {0u, 0u, 0u, 0u, 0u, 0u};
  if (role.finisher && w == 0) load_row_bits(t, y_dtype, rb * 128 + lane, raw);
  HTR_PIN();
  prefetch(buf[0]);
  if (active) {
#pragma unroll
    for (int uf = 0; uf < 8; ++uf) load_b(0, uf, 0);
  }
  prefetch(buf[1]);
  if (active) {
#pragma unroll
    for (int uf = 0; uf < 8; ++uf) load_b(1, uf, 1);
  }

  if (tid < ROWS) s_sc[tid] = tid < M ? ((const HTR_GLOBAL float*)t.sc_g)[j0 + tid] : 0.f;
  if (role.finisher && w == 0) { place_row_consts(t, raw, y_dtype, lane, consts); place_row_signs(raw, lane, consts); }

  f16v acc[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
  const int hist = history_lane_byteaddr(lane);
  // where this lane's granule goes: unit cq, piece 2 rh + strip / 2
  unsigned char* a_put = lds + ((cq * 8 + 2 * rh + ((l32 >> 3) >> 1)) * 64 + kg * 32 + ((l32 >> 3) & 1) * 8 + (lane & 7)) * 16;
  const unsigned char* a_get = lds + lane * 16;
  // One block: the products of the operands in buffer `slot` in eight parts (16 columns each), the A operands of a part read while
  // the one before it is multiplied, an eighth of the next block's decode between its matrix instructions, and the
  // activations of the block after next requested into the registers it leaves.
  auto step = [&](int slot, int v, bool more, auto active_c, StreamRegs<K>& sr) {
    constexpr bool ACTIVE = decltype(active_c)::value;
    h8 fa[2][4];
    auto fetch = [&](int uf) {
#pragma unroll
      for (int b = 0; b < 4; ++b) fa[uf & 1][b] = *(const h8*)(a_get + slot * WIDE_A + (uf * 4 + b) * 1024);
    };
    if constexpr (ACTIVE) fetch(0);
    Window<K> win;
    uint32_t prev = 0u;
    unsigned char* put = a_put + (slot ^ 1) * WIDE_A;
    if (more) {
      prev = (uint32_t)__builtin_amdgcn_ds_bpermute(hist, (int)sr.d[K - 1]);
      win.build_tail(sr);
    }
    auto pair = [&](auto u_c) { return centred(win.template pair_f16<decltype(u_c)::value>()); };
    u4 d;
#pragma unroll
    for (int uf = 0; uf < 8; ++uf) {
      if (ACTIVE && uf < 7) fetch(uf + 1);
      HTR_PIN();
      if (more) {
        // the decode touches no memory: without these pins the compiler does all of it ahead of the matrix instructions
#pragma unroll
        for (int k = 1; k <= K; ++k) asm volatile("" : "+v"(win.V[k]));
#pragma unroll
        for (int k = 1; k < K; ++k) asm volatile("" : "+v"(win.mid[k]));
        if (uf == 6) { asm volatile("" : "+v"(prev)); win.build_head(prev); }
        if (uf == 7) { asm volatile("" : "+v"(win.V[0])); asm volatile("" : "+v"(win.mid[0])); }
      }
      if constexpr (ACTIVE) {
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[uf & 1][b], B[slot][uf], acc[b], 0, 0, 0);
      }
      if (more) {
        if (uf == 0) { d.x = pair(std::integral_constant<int, 8>{}); d.y = pair(std::integral_constant<int, 10>{}); }
        if (uf == 1) { d.z = pair(std::integral_constant<int, 12>{}); d.w = pair(std::integral_constant<int, 14>{}); *(u4*)(put + 4096) = d; }            // even row, columns 8..15
        if (uf == 2) { d.x = pair(std::integral_constant<int, 16>{}); d.y = pair(std::integral_constant<int, 18>{}); }
        if (uf == 3) { d.z = pair(std::integral_constant<int, 20>{}); d.w = pair(std::integral_constant<int, 22>{}); *(u4*)(put + 256) = d; }             // odd row, columns 0..7
        if (uf == 4) { d.x = pair(std::integral_constant<int, 24>{}); d.y = pair(std::integral_constant<int, 26>{}); }
        if (uf == 5) { d.z = pair(std::integral_constant<int, 28>{}); d.w = pair(std::integral_constant<int, 30>{}); *(u4*)(put + 4096 + 256) = d; }      // odd row, columns 8..15
        if (uf == 6) { d.x = pair(std::integral_constant<int, 0>{}); d.y = pair(std::integral_constant<int, 2>{}); }
        if (uf == 7) { d.z = pair(std::integral_constant<int, 4>{}); d.w = pair(std::integral_constant<int, 6>{}); *(u4*)put = d; }                       // even row, columns 0..7
        if constexpr (ACTIVE) {
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // one matrix instruction
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);    // vector instructions
          }
        }
      }
      HTR_PIN();
      if (ACTIVE) load_b(slot, uf, v + 2);
      HTR_PIN();
    }
    if (more) prefetch(sr);
    HTR_PIN();
    __syncthreads();
    HTR_PIN();
  };
  auto run = [&](auto active_c) {
    int v = 0;
    for (; v + P < nsteps; v += P) {
#pragma unroll
      for (int pp = 0; pp < P; ++pp) step(pp, v + pp, true, active_c, buf[(pp + 1) % P]);
    }
#pragma unroll
    for (int pp = 0; pp < P; ++pp)
      if (v + pp < nsteps) step(pp, v + pp, v + pp + 1 < nsteps, active_c, buf[(pp + 1) % P]);
  };
  {
    DecodedStep<K> d0;
    decode_step<K>(buf[0], hist, d0);
    prefetch(buf[0]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      u4 q = __builtin_bit_cast(u4, d0.a[k]);
      q = u4{centred(q.x), centred(q.y), centred(q.z), centred(q.w)};
      *(u4*)(a_put + (k & 1) * 4096 + (k >> 1) * 256) = q;
    }
  }
  __syncthreads();
  if (active) run(std::true_type{}); else run(std::false_type{});

  // ---- output: lane holds activation row 32 w + lane % 32; register r of the 32 x 32 piece b is row i = 8 (r / 4) + 4 kg + r % 4 =
  // 16 x parity + 8 x strip parity + row pair, so the registers of both parities interleave to 8 consecutive weight rows
  if (active) {
    const int j = w * 32 + l32;
    const float sc = s_sc[j];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      float* dst = s_fin + j * TILE_FIN_LD + 32 * b + 8 * kg;
#pragma unroll
      for (int sl = 0; sl < 2; ++sl) {
        const f4 lo = {acc[b][4 * sl] * sc, acc[b][8 + 4 * sl] * sc, acc[b][4 * sl + 1] * sc, acc[b][8 + 4 * sl + 1] * sc};
        const f4 hi = {acc[b][4 * sl + 2] * sc, acc[b][8 + 4 * sl + 2] * sc, acc[b][4 * sl + 3] * sc, acc[b][8 + 4 * sl + 3] * sc};
        *(f4*)(dst + 16 * sl) = lo;
        *(f4*)(dst + 16 * sl + 4) = hi;
      }
    }
  }
  __syncthreads();
  const uint32_t stale = load_status(t.status);                  // non-zero: an earlier launch on this workspace gave up
  void* y = (unsigned char*)t.y + (size_t)j0 * m * (y_dtype == HTR_F32 ? 4 : 2);
  finish_tile<false, false>(t, y, part + (size_t)id0 * ROWS * 128, rb, m, M, role, s_fin, 0, consts, stale, w, lane, y_dtype);
}
