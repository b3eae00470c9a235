// Part of htr_gfx950.hip, included inside its anonymous namespace: k_viterbi: the encoder's trellis search.
// ------------------------------------------------------------------------------------------------ encoder search
// Tail-biting bitshift-trellis Viterbi over the 65536 codec states (htr/reference.py:6-50 of the reference; its GPU
// versions are htr/vit_v1.py and htr/vit_v2.py): per 256-weight tile, minimise sum_t w_t (x_t - cb[s_t])^2 with
// s_t = ((s_{t-1} << K) & 0xFFFF) | bits.  One workgroup works on one tile at a time.  Only the minima over the 2^K
// predecessors, M_t[low] = min_j cost_{t-1}[j * Sj + low] (Sj = 65536 >> K entries), need to live between steps, and
// cost_t[s] = M_t[s >> K] + w_t (x_t - cb[s])^2, so two M arrays in LDS carry a whole tile (128 KB at K2, 32 KB at K4)
// and no cost array ever goes to memory.
// A thread owns 64 states for the whole launch and keeps their codebook values in registers over a tile's passes (1024 threads x 64 = all
// 65536), so a candidate costs a subtraction, two multiplications and an addition, which this chip issues every 2.35
// cycles from vector registers, and half a v_min3 (4.2).  (Looking the penalty up in a 1021-entry LDS table, as the first
// version did, costs 5.4 cycles of the one LDS per 64 candidates plus the address arithmetic at the 4.2-cycle rate; even an eighth
// of them from a table made two steps ahead, without that arithmetic, is 4 % slower than none: the M values are read through LDS too.)
// The forward passes keep no backpointers at all: comparing and selecting an index costs 8.4 cycles per candidate against
// 2.1 for the minimum alone.  Instead the deciding pass writes every C-th M array to memory, and the trace back
// recomputes the C steps in between for the predecessors of the ONE state it is at (2^(K C) entries of M_{t-C}, 32 to 512
// of them, one wave), with the same arithmetic, so the indices it finds are those the forward pass would have recorded.
// Which array comes next does not depend on the state, so the other waves fetch it into LDS meanwhile.
// Bound: vector issue in the forward passes (K4: 2890 cycles a step, 2944 by the rates above; 0.74 M cycles a pass), then
// the trace back, 10 % of a tile at K3 and K4: its stored arrays (2 MB a tile), then one wave's chain of LDS reads and lane
// minima.  C: a larger one stores less and recomputes more (176 tiles, C - 1 instead: K2 929 us for 898, K3 823 / 763, K4 812 / 732).
// Registers: the codebook values are read anew for every tile, so that the trace back has their registers.  20 of a lane's lay in
// scratch at K4, and loading them in every turn waited for all arrays in flight.  From K3 on its loop now loads nothing from scratch;
// at K2, where 16 elements of an array are a lane's, it still loads seven registers in two turns.  Scratch bytes of a lane at K2 to K8:
// 108, 60, 44, 68, 64, 404, 140 (332, 116, 68, 44, 36, 404, 136 then), loaded once a tile or once a pass, never in the steps.  176 tiles, one per CU, us at K2 to K8: 1226, 829, 823, 956, 850, 1078, 974 before, 979, 772, 743,
// 858, 833, 895, 844 now; 1024 at K4 3.25 -> 3.03 ms (7.46 with the table and one byte of backpointer per entry and step, the first
// version).
// Arithmetic and tie-breaking are the reference's: float32, d = (x - cb)^2, m + w * d without fusing, the first index
// among equal values in every min / argmin.
template <int K> struct VitCfg {
  static constexpr int NB = 1 << K, SJ = 65536 >> K, PB = SJ / NB;
  static constexpr int THREADS = 1024;
  static constexpr int LOWS = SJ >= THREADS ? SJ / THREADS : 1;       // M entries of a thread, in runs of consecutive ones
  static constexpr int RUN = LOWS < NB ? (LOWS < 8 ? LOWS : 8) : (NB < 8 ? NB : 8), RUNS = LOWS / RUN;
  static constexpr int LANES = SJ >= THREADS ? 1 : THREADS / SJ;      // threads that share one M entry (K = 7, 8)
  static constexpr int NJ = NB / LANES;                               // predecessors a thread looks at: LOWS * NJ = 64
  static constexpr int C = K == 2 ? 4 : (K == 3 ? 3 : (K == 4 ? 2 : 1));  // steps per stored M array
  static constexpr int ROW = SJ + SJ / 16;                            // floats of an M array in LDS (the trace back shifts every 16)
  static constexpr size_t LDS = ((size_t)2 * ROW + 1024 + 512 + 32 + 128) * 4;
};
// stored M arrays of one tile: M_t for t = T - 1 - C, T - 1 - 2 C, ... > 0
inline __host__ __device__ int vit_rows(int T, int C) { return T >= 2 ? (T - 2) / C : 0; }

// one stage of an argmin over lanes: (v, k) becomes the better of this lane's and lane ^ H's, the smaller k among equals
template <int H> __device__ __forceinline__ void argmin_stage(float& v, uint32_t& k) {
  if constexpr (H <= 8) {
    const float ov = lane_xor_dpp<H>(v);
    const uint32_t ok = __float_as_uint(lane_xor_dpp<H>(__uint_as_float(k)));
    if (ov < v || (ov == v && ok < k)) { v = ov; k = ok; }
  } else {
    const uint32_t u = __float_as_uint(v);
    u2s rv, rk;
    if constexpr (H == 16) { rv = __builtin_amdgcn_permlane16_swap(u, u, false, false); rk = __builtin_amdgcn_permlane16_swap(k, k, false, false); }
    else { rv = __builtin_amdgcn_permlane32_swap(u, u, false, false); rk = __builtin_amdgcn_permlane32_swap(k, k, false, false); }
    const float a = __uint_as_float(rv.x), b = __uint_as_float(rv.y);
    const bool second = b < a || (b == a && rk.y < rk.x);
    v = second ? b : a; k = second ? rk.y : rk.x;
  }
}
template <int SPAN> __device__ __forceinline__ void argmin_lanes(float& v, uint32_t& k) {      // over groups of SPAN adjacent lanes
  if constexpr (SPAN >= 2) argmin_stage<1>(v, k);
  if constexpr (SPAN >= 4) argmin_stage<2>(v, k);
  if constexpr (SPAN >= 8) argmin_stage<4>(v, k);
  if constexpr (SPAN >= 16) argmin_stage<8>(v, k);
  if constexpr (SPAN >= 32) argmin_stage<16>(v, k);
  if constexpr (SPAN >= 64) argmin_stage<32>(v, k);
}

template <int K>
__global__ __launch_bounds__(VitCfg<K>::THREADS) void k_viterbi(const float* __restrict__ x, const float* __restrict__ w, int tiles,
                                                               int T, int tailbite, float* __restrict__ rows_g,
                                                               uint16_t* __restrict__ states, double rms) {
#pragma clang fp contract(off)          // m + w d^2 stays a multiplication and an addition (the __f*_rn functions do not keep the compiler from fusing)
  using V = VitCfg<K>;
  constexpr int SJ = V::SJ, PB = V::PB, THREADS = V::THREADS, RUN = V::RUN, RUNS = V::RUNS, LANES = V::LANES,
                NJ = V::NJ, C = V::C;
  extern __shared__ __align__(16) unsigned char lds[];
  float* M0 = (float*)lds;                 // [ROW]
  float* M1 = M0 + V::ROW;                 // [ROW]
  float* cbv = M1 + V::ROW;                // [1024] codebook value of each v
  float* xs = cbv + 1024;                  // [256] targets, [256] weights
  float* ws = xs + 256;
  float* red_v = ws + 256;                 // [16] reduction scratch
  uint32_t* red_i = (uint32_t*)(red_v + 16);
  const int tid = threadIdx.x, lane = tid & 63;
  // this thread's M entries low(r, i) and predecessors pj(j)
  auto low_of = [](int r, int i, int id) { return LANES == 1 ? (r * THREADS + id) * RUN + i : id / LANES; };
  auto pj_of = [](int j, int id) { return LANES == 1 ? j : j * LANES + id % LANES; };
  auto low = [&](int r, int i) { return low_of(r, i, tid); };
  auto pj = [&](int j) { return pj_of(j, tid); };

  for (int i = tid; i < 1024; i += THREADS) cbv[i] = i <= 1020 ? (float)((double)(i - 510) / rms) : 0.f;
  __syncthreads();
  auto cb_of = [&](uint32_t s) { return cbv[__builtin_amdgcn_sad_u8(s * GEN_A + GEN_B, 0u, 0u)]; };
  const int nrows = vit_rows(T, C);
  float* my_rows = rows_g + (size_t)blockIdx.x * nrows * SJ;          // one set of stored arrays per workgroup, reused tile by tile
  for (size_t tile = blockIdx.x; tile < (size_t)tiles; tile += gridDim.x) {
    for (int i = tid; i < T; i += THREADS) { xs[i] = x[tile * T + i]; ws[i] = w[tile * T + i]; }
    // the codebook values of this thread's states: read again for every tile (2 us of 800), so that the trace back has their registers
    float cb[RUNS][RUN][NJ];
    int own = tid;
    asm volatile("" : "+v"(own));                         // or the compiler keeps the 64 addresses over the trace back instead
#pragma unroll
    for (int r = 0; r < RUNS; ++r)
#pragma unroll
      for (int i = 0; i < RUN; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) cb[r][i][j] = cb_of((uint32_t)(pj_of(j, own) * SJ + low_of(r, i, own)));
    uint32_t j0 = 0, final_state = 0;
    const int passes = tailbite ? 2 : 1;
    for (int pass = 0; pass < passes; ++pass) {
      const bool constrained = pass == 1;             // second pass: start and end tied to j0
      const bool record = pass == passes - 1;
      // cost_0[s] = M_0[s >> K] + term_0(s) with M_0 = 0 (free start) or 0 at j0 and infinity elsewhere
      for (int i = tid; i < SJ; i += THREADS) M0[i] = (!constrained || (uint32_t)i == j0) ? 0.f : __builtin_inff();
      __syncthreads();
      float* Mold = M0;
      float* Mnew = M1;
      int until = T - 2 < 0 ? 0 : (T - 2) % C;         // steps until the next stored array: M_{t+1} with (T - 2 - t) % C == 0
      float* row = my_rows;
      for (int t = 0; t < T - 1; ++t) {
        const float xt = xs[t], wt = ws[t];
        const bool keep = record && until == 0 && t + 1 < T - 1;
#pragma unroll
        for (int r = 0; r < RUNS; ++r) {
          float best[RUN];
#pragma unroll
          for (int i = 0; i < RUN; ++i) best[i] = __builtin_inff();
          const float* m_in = Mold + (low(r, 0) >> K);          // a run lies inside one predecessor group
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            const float m = m_in[pj(j) * PB];
#pragma unroll
            for (int i = 0; i < RUN; ++i) {
              const float d = xt - cb[r][i][j];
              best[i] = fminf(best[i], m + wt * (d * d));
            }
          }
          if constexpr (LANES >= 2) best[0] = fminf(best[0], lane_xor_dpp<1>(best[0]));
          if constexpr (LANES >= 4) best[0] = fminf(best[0], lane_xor_dpp<2>(best[0]));
          float* m_out = Mnew + low(r, 0);
          float* g_out = row + low(r, 0);
          if constexpr (RUN % 4 == 0) {
#pragma unroll
            for (int i = 0; i < RUN; i += 4) {
              const f4 q = {best[i], best[i + 1], best[i + 2], best[i + 3]};
              *(f4*)(m_out + i) = q;
              if (keep) *(f4*)(g_out + i) = q;
            }
          } else if (LANES == 1 || tid % LANES == 0) {
#pragma unroll
            for (int i = 0; i < RUN; ++i) {
              m_out[i] = best[i];
              if (keep) g_out[i] = best[i];
            }
          }
        }
        if (keep) row += SJ;
        until = until == 0 ? C - 1 : until - 1;
        __syncthreads();
        float* tmp = Mold; Mold = Mnew; Mnew = tmp;
      }
      // last step: argmin over all states of cost_{T-1}, first index among equals; second pass: only states whose
      // lower part is j0
      const float xt = xs[T - 1], wt = ws[T - 1];
      float best = __builtin_inff();
      uint32_t bs = 0xFFFFFFFFu;
#pragma unroll
      for (int r = 0; r < RUNS; ++r)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const float m = Mold[pj(j) * PB + (low(r, 0) >> K)];
#pragma unroll
          for (int i = 0; i < RUN; ++i) {
            const uint32_t s = (uint32_t)(pj(j) * SJ + low(r, i));
            const float d = xt - cb[r][i][j];
            float c = m + wt * (d * d);
            if (constrained && (uint32_t)low(r, i) != j0) c = __builtin_inff();
            if (c < best || (c == best && s < bs)) { best = c; bs = s; }
          }
        }
      // wave, then workgroup reduction of (value, index)
      argmin_lanes<64>(best, bs);
      if (lane == 0) { red_v[tid >> 6] = best; red_i[tid >> 6] = bs; }
      __syncthreads();
      float b = red_v[lane & 15];
      uint32_t bi = red_i[lane & 15];
      argmin_lanes<16>(b, bi);
      final_state = bi == 0xFFFFFFFFu ? 0u : bi;        // every cost infinite or NaN: the reference's argmin gives 0
      __syncthreads();
      if (!record) j0 = final_state & (SJ - 1);
    }
    // ---- trace back (htr/reference.py:43-49): from s_t to s_{t-1} .. s_{t-n}, n = min(C, t), in one turn.  With p_0 = s_t >> K
    // and predecessors j_1, j_2, .., the state s_{t-d-1} is (j_{d+1}, p_d), p_d = (j_d, .., j_1, upper bits of p_0), and
    // M_{t-d}[p_d] = min over j_{d+1} of M_{t-d-1}[(j_{d+1}, p_d) >> K] + term.  A lane stands for one (j_n, .., j_1), j_n in its
    // lowest bits (and the upper bits of j_n, if the lanes do not suffice, in PER registers): level n - 1 reads M_{t-n},
    // each level is a minimum over the lanes of one digit, which leaves the next level's values where they are needed.
    // The lanes that attain a level's minimum are kept as a mask, and the digits are read off the masks at the end.
    uint16_t* st = (uint16_t*)red_v + 64;               // [256] in LDS, out at the end
    if (tid == 0) st[T - 1] = (uint16_t)final_state;
    if (T > 1) {
      // in registers of their own: what the compiler derives from them and keeps is not kept over the forward passes
      int id = tid, ln = lane;
      asm volatile("" : "+v"(id), "+v"(ln));
      constexpr int RL = SJ >= THREADS ? SJ / THREADS : 1;             // row elements per thread
      auto lds_pos = [](uint32_t e) { return e + (e >> 4); };
      // The q-th array that the trace back reads: the stored ones from the last on, then M_0.  Nothing in the loop may make it wait for
      // loads that it has just issued: no branch around a load (M_0 comes in where the array goes to LDS), from K3 on no value in scratch.
      auto request = [&](float (&reg)[RL], int q) {                    // beyond the last stored one: the first again, not looked at
        const float* row = my_rows + (size_t)max(nrows - 1 - q, 0) * SJ;
#pragma unroll
        for (int i = 0; i < RL; ++i) reg[i] = row[(i * THREADS + id) & (SJ - 1)];
      };
      auto place = [&](const float (&reg)[RL], int q, float* buf) {
        auto first = [&](uint32_t e) { return !tailbite || e == j0 ? 0.f : __builtin_inff(); };      // M_0
#pragma unroll
        for (int i = 0; i < RL; ++i) {
          const uint32_t e = (uint32_t)(i * THREADS + id);
          if (SJ >= THREADS || id < SJ) buf[lds_pos(e)] = RL > 8 || q < nrows ? reg[i] : first(e);
        }
        // with 16 elements a thread the selections above would take longer than a second pass at the end (176 tiles at K2, 966 / 900 us)
        if (RL > 8 && q >= nrows)
          for (int e = id; e < SJ; e += THREADS) buf[lds_pos((uint32_t)e)] = first((uint32_t)e);
      };
      uint32_t s = final_state;
      auto turn = [&](auto nc, const float* buf, int t) {
        constexpr int n = decltype(nc)::value;
        constexpr int PERB = K * n > 6 ? K * n - 6 : 0, PER = 1 << PERB, NBITS = K - PERB;      // lane bits of j_n
        const uint32_t p0 = s >> K;
        auto digit = [&](int i) { return i == n ? (uint32_t)ln & ((1u << NBITS) - 1) : ((uint32_t)ln >> (NBITS + K * (n - 1 - i))) & ((1u << K) - 1); };
        unsigned long long mask[n][PER];
        float v = 0.f;
#pragma unroll
        for (int d = n - 1; d >= 0; --d) {
          uint32_t p = p0 >> (K * d);
#pragma unroll
          for (int i = 1; i <= d; ++i) p |= digit(i) << (16 - K - K * (d - i + 1));
          const float xt = xs[t - d - 1], wt = ws[t - d - 1];
          float c[PER];
          const int per = d == n - 1 ? PER : 1;
#pragma unroll
          for (int k = 0; k < per; ++k) {
            const uint32_t state = ((digit(d + 1) | (d == n - 1 ? (uint32_t)k << NBITS : 0u)) << (16 - K)) | p;
            const float m = d == n - 1 ? buf[lds_pos(state >> K)] : v;
            const float dd = xt - cb_of(state);
            c[k] = m + wt * (dd * dd);
          }
          v = c[0];
#pragma unroll
          for (int k = 1; k < per; ++k) v = fminf(v, c[k]);
          // over the lane bits of digit d + 1; the lower bits hold equal values already, so a mirror is as good as an xor
          const int lo = d == n - 1 ? 0 : NBITS + K * (n - 2 - d), hi = d == n - 1 ? NBITS : lo + K;
#pragma unroll
          for (int bit = lo; bit < hi; ++bit) {
            if (bit == 0) v = fminf(v, dpp_mov<0xB1>(v));
            if (bit == 1) v = fminf(v, dpp_mov<0x4E>(v));
            if (bit == 2) v = fminf(v, dpp_mov<0x141>(v));
            if (bit == 3) v = fminf(v, dpp_mov<0x140>(v));
            if (bit == 4) { float e, o; halves16(v, e, o); v = fminf(e, o); }
            if (bit == 5) { float e, o; halves32(v, e, o); v = fminf(e, o); }
          }
#pragma unroll
          for (int k = 0; k < per; ++k) mask[d][k] = __ballot(c[k] == v);
        }
        uint32_t base = 0u;                                            // first lane of the digits found so far
#pragma unroll
        for (int d = 0; d < n; ++d) {
          const int shift = d == n - 1 ? 0 : NBITS + K * (n - 2 - d), width = d == n - 1 ? NBITS : K;
          const int span = 1 << (shift + width);                       // lanes that share those digits
          const unsigned long long in_span = span >= 64 ? ~0ull : ((1ull << (span & 63)) - 1);
          uint32_t j = 0u;
          bool found = false;
#pragma unroll
          for (int k = 0; k < (d == n - 1 ? PER : 1); ++k) {
            const unsigned long long mk = (mask[d][k] >> base) & in_span;
            if (!found && mk != 0ull) { j = ((uint32_t)__builtin_ctzll(mk) >> shift) | ((uint32_t)k << width); found = true; }
          }
          if (d < n - 1) base += j << shift;
          s = j * SJ + (s >> K);
          if (ln == 0) st[t - d - 1] = (uint16_t)s;
        }
      };
      // arrays travel AHEAD turns ahead in registers, one more in the other LDS buffer
      constexpr int AHEAD = RL <= 8 ? 4 : 1, UNROLL = AHEAD > 2 ? AHEAD : 2;
      float set[AHEAD][RL];
      request(set[0], 0);
      place(set[0], 0, M0);
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) request(set[i], 1 + i);
      __syncthreads();
      const int full = (T - 1) / C, rest = (T - 1) % C;
      for (int k0 = 0; k0 < full; k0 += UNROLL) {
#pragma unroll
        for (int i = 0; i < UNROLL; ++i) {
          const int k = k0 + i;
          if (k >= full) break;                                        // uniform
          place(set[i % AHEAD], k + 1, i & 1 ? M0 : M1);
          request(set[i % AHEAD], k + 1 + AHEAD);
          if (id < 64) turn(std::integral_constant<int, C>{}, i & 1 ? M1 : M0, T - 1 - C * k);
          __syncthreads();
        }
      }
      if (C > 1 && rest > 0 && id < 64) {                              // from M_0 itself
        const float* buf = full & 1 ? M1 : M0;
        if (C >= 4 && rest == 3) turn(std::integral_constant<int, (C >= 4 ? 3 : 1)>{}, buf, rest);
        else if (C >= 3 && rest == 2) turn(std::integral_constant<int, (C >= 3 ? 2 : 1)>{}, buf, rest);
        else turn(std::integral_constant<int, 1>{}, buf, rest);
      }
    }
    __syncthreads();
    for (int i = tid; i < T; i += THREADS) states[tile * T + i] = st[i];
    __syncthreads();                                    // xs, ws and the M arrays are free for the next tile
  }
}

// ------------------------------------------------------------------------------------------------ around the search
// One 16-column block of the encoder's matrices before and after its search (htr/encode.py:69-88 of the reference): every thread
// takes four consecutive elements of one row.  float32 and unfused, in the reference's order of operations.
// targets: x = (W + F) / row scale, as the search wants its tiles.
__global__ __launch_bounds__(256) void k_encode_targets(const float* __restrict__ W, const float* __restrict__ F, const float* __restrict__ rs,
                                                        int64_t rows, int64_t ld, int64_t col, float* __restrict__ x) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, row = i >> 2;
  if (row >= rows) return;
  const int64_t at = row * ld + col + 4 * (i & 3);
  const f4 sum = *(const f4*)(W + at) + *(const f4*)(F + at);
  const float r = rs[row];
  *(f4*)(x + 4 * i) = f4{sum.x / r, sum.y / r, sum.z / r, sum.w / r};
}
// quantized: q = cb[s] * row scale into Q, W - q into err, the states as whole numbers into S [tile][blocks][256].  Bound: the launch;
// with the kernel above two launches of 4 us where torch takes eleven, 0.9 MB each at 2816 rows.
__global__ __launch_bounds__(256) void k_encode_quantized(const uint16_t* __restrict__ states, const float* __restrict__ cb, const float* __restrict__ W,
                                                          const float* __restrict__ rs, int64_t rows, int64_t ld, int64_t col,
                                                          float* __restrict__ Q, float* __restrict__ err, int64_t* __restrict__ S) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, row = i >> 2;
  if (row >= rows) return;
  const int64_t at = row * ld + col + 4 * (i & 3);
  const float r = rs[row];
  const f4 w = *(const f4*)(W + at);
  uint32_t s[4];
  f4 q, e;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    s[k] = states[4 * i + k];
    q[k] = cb[s[k]] * r;
    e[k] = w[k] - q[k];
  }
  *(f4*)(Q + at) = q;
  *(f4*)(err + 4 * i) = e;
  typedef int64_t l2 __attribute__((ext_vector_type(2)));
  l2* o = (l2*)(S + ((row >> 4) * (ld >> 4) + (col >> 4)) * 256 + (4 * i & 255));
  o[0] = l2{(int64_t)s[0], (int64_t)s[1]};
  o[1] = l2{(int64_t)s[2], (int64_t)s[3]};
}
