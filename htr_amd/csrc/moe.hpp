// Part of htr_gfx950.hip, included inside its anonymous namespace: routing, rotation, activation and combination around the
// two grouped launches (k_linear_tile) of a routed-expert layer.
// ------------------------------------------------------------------------------------------------ routed experts
// One layer is six launches, and no copy or synchronisation between them:
//   k_moe_route     one workgroup: tokens sorted by expert, the problem tables of both grouped launches; up to 64 experts' tensor
//                   addresses come as kernel arguments (16 tokens, 64 experts: two launches of k_moe_experts less, 4 of 76 us), more of
//                   them through a device table that k_moe_experts fills (one launch per 64 experts)
//   k_moe_rotate    one workgroup per (token, expert) pair: gather, sign, H128, f16, in fragment order
//   k_linear_tile   gate and up of every active expert, float32
//   k_moe_act       one workgroup per pair: silu(gate) * up, rounded to the activations' type, then as k_moe_rotate
//   k_linear_tile   down, float32
//   k_moe_combine   y_t = sum_j w_tj out(t, j), j ascending
// Every entry of the problem tables is one expert and up to rows_per_entry of its pairs; the number of entries is known to the
// host only as a bound (experts + pairs / rows per entry), entries beyond the used ones have no rows and their workgroups
// return at once.
constexpr int MOE_PTR_CHUNK = 64;                 // experts per launch that takes their addresses: 4 KB of kernel arguments
struct MoePtrs { const void* p[MOE_PTR_CHUNK][8]; };      // gate_up: qweight, scales, su, sv; down: the same

__global__ __launch_bounds__(MOE_PTR_CHUNK * 8) void k_moe_experts(const MoePtrs src, const void** __restrict__ table, int first, int count) {
  const int i = threadIdx.x;
  if (i < count * 8) table[first * 8 + i] = src.p[i >> 3][i & 7];
}

struct MoeRoute {
  const void* ids;               // [pairs] int32 or int64
  int ids64, pairs, top, experts, entries, rows_per_entry;
  const void** table;            // [experts][8]
  int m1, m2;                    // rows of gate_up and of down
  htr_group_entry* e1;           // [entries]
  htr_group_entry* e2;
  float* h;                      // [pairs][m1]
  float* out;                    // [pairs][m2]
  int* pos_of;                   // [pairs] (token, slot) -> sorted position
  int4* info;                    // [pairs] sorted position -> {token, expert, row of the fragment order, unused}
  uint32_t* host_word;           // pinned: ticket << 1 | some id is out of range
  uint32_t ticket;
};
// Counting sort by expert.  A pair's rank within its expert is whatever the LDS counter returns: the results do not depend on
// which row of a tile a pair occupies.  The pairs of a wave that share its first pair's expert take their ranks together
// (lanes that hit one LDS counter are served one after the other, about 64 cycles each, and a popular expert would cost
// that for every pair).
constexpr int MOE_ROUTE_THREADS = 1024;
constexpr int MOE_MAX_EXPERTS = 4096;
// GIVEN: the experts' addresses are in `ptrs` and go to the table here; otherwise they are in it
template <bool GIVEN>
__global__ __launch_bounds__(MOE_ROUTE_THREADS) void k_moe_route(const MoeRoute a, const MoePtrs ptrs) {
  __shared__ uint32_t cnt[MOE_MAX_EXPERTS];       // pairs of the expert, then its first position
  __shared__ uint32_t row0[MOE_MAX_EXPERTS];      // row of the fragment order of a pair = its position + this (mod 2^32)
  __shared__ uint32_t s_scan[3][16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int E = a.experts, R = a.rows_per_entry;
  auto id_of = [&](int p) {
    const long long v = a.ids64 ? ((const long long*)a.ids)[p] : (long long)((const int*)a.ids)[p];
    return v < 0 || v >= E ? -1 : (int)v;
  };
  for (int i = tid; i < E; i += MOE_ROUTE_THREADS) cnt[i] = 0u;
  if (GIVEN && tid < E * 8) a.table[tid] = ptrs.p[tid >> 3][tid & 7];
  __syncthreads();
  bool bad = false;
  for (int q0 = w * 64; q0 < a.pairs; q0 += MOE_ROUTE_THREADS) {
    const int p = q0 + lane;
    const int e = p < a.pairs ? id_of(p) : -1;
    bad |= p < a.pairs && e < 0;
    const int first = __builtin_amdgcn_readfirstlane(e);
    const unsigned long long same = __ballot(e == first);
    uint32_t rank = 0u;
    if (e >= 0 && e != first) rank = atomicAdd(&cnt[e], 1u);
    if (first >= 0) {
      uint32_t base = 0u;
      if (lane == 0) base = atomicAdd(&cnt[first], (uint32_t)__builtin_popcountll(same));
      base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
      if (e == first) rank = base + (uint32_t)__builtin_popcountll(same & ((1ull << lane) - 1ull));
    }
    if (p < a.pairs) a.pos_of[p] = (int)rank;
  }
  bad = __syncthreads_or(bad);
  if (tid == 0 && a.host_word != nullptr)
    __hip_atomic_store(a.host_word, (a.ticket << 1) | (bad ? 1u : 0u), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  // prefix over the experts of pairs, table entries and 32-row tiles; the tables
  uint32_t pos_base = 0u, ent_base = 0u, tile_base = 0u;
  for (int e0 = 0; e0 < E; e0 += MOE_ROUTE_THREADS) {
    const int e = e0 + tid;
    const uint32_t total = e < E ? cnt[e] : 0u, ents = (total + R - 1) / R, tiles = (total + 31) / 32;
    uint32_t a0 = total, a1 = ents, a2 = tiles;    // inclusive scans over the wave
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t b0 = __shfl_up(a0, off), b1 = __shfl_up(a1, off), b2 = __shfl_up(a2, off);
      if (lane >= off) { a0 += b0; a1 += b1; a2 += b2; }
    }
    if (lane == 63) { s_scan[0][w] = a0; s_scan[1][w] = a1; s_scan[2][w] = a2; }
    __syncthreads();
    uint32_t w0 = 0u, w1 = 0u, w2 = 0u, t0 = 0u, t1 = 0u, t2 = 0u;
    for (int k = 0; k < MOE_ROUTE_THREADS / 64; ++k) {
      if (k < w) { w0 += s_scan[0][k]; w1 += s_scan[1][k]; w2 += s_scan[2][k]; }
      t0 += s_scan[0][k]; t1 += s_scan[1][k]; t2 += s_scan[2][k];
    }
    const uint32_t pos = pos_base + w0 + a0 - total, ent = ent_base + w1 + a1 - ents, tile = tile_base + w2 + a2 - tiles;
    if (e < E) {
      cnt[e] = pos;
      row0[e] = tile * 32u - pos;
      const void* t[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) t[k] = GIVEN ? ptrs.p[e][k] : a.table[(size_t)e * 8 + k];
      for (uint32_t i = 0; i < ents; ++i) {
        const uint32_t r0 = i * R, rows = min((uint32_t)R, total - r0);
        htr_group_entry g;
        g.bias = nullptr; g.x = nullptr; g.M = (int)rows; g.reserved = (int)(tile + r0 / 32u);      // R is a multiple of 32
        g.qweight = t[0]; g.scales = t[1]; g.su = t[2]; g.sv = t[3]; g.y = a.h + (size_t)(pos + r0) * a.m1;
        a.e1[ent + i] = g;
        g.qweight = t[4]; g.scales = t[5]; g.su = t[6]; g.sv = t[7]; g.y = a.out + (size_t)(pos + r0) * a.m2;
        a.e2[ent + i] = g;
      }
    }
    pos_base += t0; ent_base += t1; tile_base += t2;
    __syncthreads();
  }
  for (int i = (int)ent_base + tid; i < a.entries; i += MOE_ROUTE_THREADS) { a.e1[i].M = 0; a.e2[i].M = 0; }
  for (int p = tid; p < a.pairs; p += MOE_ROUTE_THREADS) {
    const int e = id_of(p);
    // a pair whose expert is out of range: not a number in the result of its token
    const int pos = e < 0 ? -1 : (int)(cnt[e] + (uint32_t)a.pos_of[p]);
    a.pos_of[p] = pos;
    if (e >= 0) a.info[pos] = int4{p / a.top, e, (int)((uint32_t)pos + row0[e]), 0};
  }
  // with such pairs the sorted list is shorter than the grids assume
  for (int p = (int)pos_base + tid; p < a.pairs; p += MOE_ROUTE_THREADS) a.info[p] = int4{0, -1, 0, 0};
}

// ---- rotation of one activation row of n elements into the fragment order, by one workgroup of 256 threads (four waves x
// four blocks a pass).  `get` returns the eight consecutive 16-bit elements from column c on.
template <typename Get>
__device__ __forceinline__ void rotate_row_frag16(Get&& get, const uint8_t* __restrict__ su, int n, bool is_bf16, size_t frow,
                                                  _Float16* __restrict__ xt_g, float* __restrict__ xs_g, float* __restrict__ sc_g,
                                                  uint32_t* s_amax) {
  constexpr int WAVES = 4, KEEP = 4;                             // passes whose elements stay in registers between the two loops
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, gk = lane >> 4, j = lane & 15, nblk = n >> 7;
  auto col_of = [&](int pass) { return ((pass * WAVES + w) * 4 + (j >> 2)) * 128 + 32 * (j & 3) + 8 * gk; };
  const int passes = (nblk + 4 * WAVES - 1) / (4 * WAVES);
  u4 xr[KEEP];
  uint32_t sb[KEEP];
  uint32_t m16 = 0u;
  auto fold = [&](const u4& v) {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) m16 = max(m16, max(d[k] & 0x7FFFu, (d[k] >> 16) & 0x7FFFu));
  };
  const u4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int p = 0; p < KEEP; ++p) {
    const int c = col_of(p);
    xr[p] = p < passes && c < n ? get(c) : zero;
    sb[p] = p < passes && c < n ? (uint32_t)su[c >> 3] : 0u;
  }
#pragma unroll
  for (int p = 0; p < KEEP; ++p) fold(xr[p]);
  for (int p = KEEP; p < passes; ++p) { const int c = col_of(p); if (c < n) fold(get(c)); }
  m16 = wave_max_u32(m16);
  if (lane == 0) s_amax[w] = m16;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < WAVES; ++k) m16 = max(m16, s_amax[k]);
  float amax = is_bf16 ? bf16_bits_to_float((uint16_t)m16) : f16_bits_to_float((uint16_t)m16);
  if (amax != amax) amax = __uint_as_float(0x7F800000u);         // a NaN anywhere: treat the row as unbounded (scale 1)
  const int e = scale_exponent(amax);
  const float f = pow2f(-e) * INV_SQRT128;
  if (threadIdx.x == 0) sc_g[frow] = pow2f(e);
  auto pass = [&](int p, const u4& x4, uint32_t bits) {
    const int b0 = (p * WAVES + w) * 4;
    if (b0 >= nblk) return;                                      // uniform per wave
    float y[2][4];
    rotate4_mfma(x4, bits, is_bf16, lane, y);
    const int blk = b0 + gk;                                     // lane (p = lane / 16, j) holds elements 32 a + 16 h + j of block b0 + p
    const bool live = blk < nblk;
    // element 32 a + 16 h + j: unit 4 blk + a, half j / 8, lane 32 h + row % 32, element j % 8
    HTR_GLOBAL _Float16* dst = (HTR_GLOBAL _Float16*)xt_g + frag_half(n, frow, blk * 128 + j);
    float r[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const _Float16 hv = (_Float16)(y[h][a] * f);
        if (live) dst[a * 1024 + h * 256] = hv;
        r[h][a] = (float)hv;
      }
    f4 sm = {(r[0][0] + r[0][1]) + (r[0][2] + r[0][3]), (r[1][0] + r[1][1]) + (r[1][2] + r[1][3]),
             (r[0][0] + r[0][1]) + (r[1][0] + r[1][1]), (r[0][2] + r[0][3]) + (r[1][2] + r[1][3])};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      float v = sm[c];
      v += dpp_mov<0xB1>(v); v += dpp_mov<0x4E>(v); v += dpp_mov<0x141>(v); v += dpp_mov<0x140>(v);
      sm[c] = v;
    }
    if (live && j == 0) *(HTR_GLOBAL f4*)((HTR_GLOBAL float*)xs_g + (frow * nblk + blk) * 4) = sm;
  };
#pragma unroll
  for (int p = 0; p < KEEP; ++p) if (p < passes) pass(p, xr[p], sb[p]);
  for (int p = KEEP; p < passes; ++p) {
    const int c = col_of(p);
    pass(p, c < n ? get(c) : zero, c < n ? (uint32_t)su[c >> 3] : 0u);
  }
}
// The same for float32 elements: `get` returns element c; butterflies over the lanes, one block per wave and pass.
template <typename Get>
__device__ __forceinline__ void rotate_row_frag32(Get&& get, const uint8_t* __restrict__ su, int n, size_t frow, _Float16* __restrict__ xt_g,
                                                  float* __restrict__ xs_g, float* __restrict__ sc_g, uint32_t* s_amax) {
  constexpr int WAVES = 4;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nblk = n >> 7;
  uint32_t m32 = 0u;
  for (int c = threadIdx.x; c < n; c += 64 * WAVES) m32 = max(m32, __float_as_uint(get(c)) & 0x7FFFFFFFu);
  m32 = wave_max_u32(m32);
  if (lane == 0) s_amax[w] = m32;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < WAVES; ++k) m32 = max(m32, s_amax[k]);
  float amax = __uint_as_float(m32);
  if (amax != amax) amax = __uint_as_float(0x7F800000u);
  const int e = scale_exponent(amax);
  const float inv = pow2f(-e);
  if (threadIdx.x == 0) sc_g[frow] = pow2f(e);
  for (int blk = w; blk < nblk; blk += WAVES) {
    const int ca = blk * 128 + lane, cb = ca + 64;
    float va = get(ca) * (((su[ca >> 3] >> (ca & 7)) & 1) ? -inv : inv), vb = get(cb) * (((su[cb >> 3] >> (cb & 7)) & 1) ? -inv : inv);
    fwht128_wave(va, vb, lane);
    const _Float16 ha = (_Float16)(va * INV_SQRT128), hb = (_Float16)(vb * INV_SQRT128);
    xt_g[frag_half(n, frow, ca)] = ha;
    xt_g[frag_half(n, frow, cb)] = hb;
    float ea, oa, eb, ob;
    wave_sum_by_row_parity((float)ha, ea, oa);
    wave_sum_by_row_parity((float)hb, eb, ob);
    if (lane == 0) *(f4*)(xs_g + (frow * nblk + blk) * 4) = f4{ea + eb, oa + ob, ea + oa, eb + ob};
  }
}

// Sorted position of the pair that a workgroup rotates.  Eight rows of an expert share every 128-byte line of the fragment order, 16
// bytes each, and workgroups go to the eight XCDs in turn, each with an L2 of its own: an eighth of the consecutive positions
// to every XCD, so that its L2 puts the lines together.  Bound of both rotations: memory latency and these writes.  500 tokens over 64
// experts (2048x1408), whole layer: 189.7 -> 185 us; 16 tokens level.
constexpr int MOE_XCDS = 8;
__host__ __device__ inline int moe_rotate_grid(int pairs) { return (pairs + MOE_XCDS - 1) / MOE_XCDS * MOE_XCDS; }
__device__ __forceinline__ int moe_pair_of(int block, int grid) { return (block % MOE_XCDS) * (grid / MOE_XCDS) + block / MOE_XCDS; }

__global__ __launch_bounds__(256) void k_moe_rotate(const void* __restrict__ x, int x_dtype, int pairs, const int4* __restrict__ info,
                                                    const void* const* __restrict__ table, int n, _Float16* __restrict__ xt_g,
                                                    float* __restrict__ xs_g, float* __restrict__ sc_g) {
  __shared__ uint32_t s_amax[4];
  const int pos = moe_pair_of(blockIdx.x, moe_rotate_grid(pairs));
  if (pos >= pairs) return;
  const int4 q = info[pos];                                      // uniform
  if (q.y < 0) return;
  const uint8_t* su = (const uint8_t*)table[(size_t)q.y * 8 + 2];
  if (x_dtype == HTR_F32) {
    const float* row = (const float*)x + (size_t)q.x * n;
    rotate_row_frag32([&](int c) { return row[c]; }, su, n, (size_t)q.z, xt_g, xs_g, sc_g, s_amax);
  } else {
    const uint16_t* row = (const uint16_t*)x + (size_t)q.x * n;
    rotate_row_frag16([&](int c) { return *(const u4*)(row + c); }, su, n, x_dtype == HTR_BF16, (size_t)q.z, xt_g, xs_g, sc_g, s_amax);
  }
}

// silu(gate) * up of one pair, rounded to the activations' type, rotated for the down projection
__global__ __launch_bounds__(256) void k_moe_act(const float* __restrict__ h, int x_dtype, int pairs, const int4* __restrict__ info,
                                                 const void* const* __restrict__ table, int F, _Float16* __restrict__ xt_g,
                                                 float* __restrict__ xs_g, float* __restrict__ sc_g) {
  __shared__ uint32_t s_amax[4];
  const int pos = moe_pair_of(blockIdx.x, moe_rotate_grid(pairs));
  if (pos >= pairs) return;
  const int4 q = info[pos];
  if (q.y < 0) return;
  const uint8_t* su = (const uint8_t*)table[(size_t)q.y * 8 + 6];
  const float* gate = h + (size_t)pos * 2 * F;
  const float* up = gate + F;
  auto act = [](float g, float u) { return g / (1.f + expf(-g)) * u; };
  if (x_dtype == HTR_F32) {
    rotate_row_frag32([&](int c) { return act(gate[c], up[c]); }, su, F, (size_t)q.z, xt_g, xs_g, sc_g, s_amax);
  } else {
    const bool is_bf16 = x_dtype == HTR_BF16;
    auto pack = [&](float a, float b) {
      if (is_bf16) return (uint32_t)float_to_bf16_bits(a) | ((uint32_t)float_to_bf16_bits(b) << 16);
      return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)a) | ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)b) << 16);
    };
    auto get = [&](int c) {
      const f4 g0 = *(const f4*)(gate + c), g1 = *(const f4*)(gate + c + 4), u0 = *(const f4*)(up + c), u1 = *(const f4*)(up + c + 4);
      return u4{pack(act(g0.x, u0.x), act(g0.y, u0.y)), pack(act(g0.z, u0.z), act(g0.w, u0.w)),
                pack(act(g1.x, u1.x), act(g1.y, u1.y)), pack(act(g1.z, u1.z), act(g1.w, u1.w))};
    };
    rotate_row_frag16(get, su, F, is_bf16, (size_t)q.z, xt_g, xs_g, sc_g, s_amax);
  }
}

// y[token] = sum over its slots, ascending; a slot without a valid expert gives NaN
__global__ __launch_bounds__(256) void k_moe_combine(const float* __restrict__ out, const int* __restrict__ pos_of, const float* __restrict__ wt,
                                                     int top, int H, float* __restrict__ y) {
  const int token = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * 4;      // tokens in x, the grid's only dimension beyond 65535
  if (c >= H) return;
  f4 s = {0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j < top; ++j) {
    const int p = pos_of[token * top + j];                       // uniform
    const float wj = p < 0 ? __builtin_nanf("") : wt[token * top + j];
    const f4 v = *(const f4*)(out + (size_t)(p < 0 ? 0 : p) * H + c);
    s += v * wj;
  }
  *(f4*)(y + (size_t)token * H + c) = s;
}
