// Part of htr_gfx950.hip, included inside its anonymous namespace: k_decode_raw, k_dequant_q, k_dequant_w.
// ------------------------------------------------------------------------------------------------ debug decodes
template <int K, int U> struct ForEach32 {
  template <typename F> __device__ __forceinline__ static void run(const Window<K>& w, F&& f) {
    f(U, w.template value<U>());
    if constexpr (U + 1 < 32) ForEach32<K, U + 1>::run(w, f);
  }
};

template <int K>
__global__ __launch_bounds__(256) void k_decode_raw(const uint32_t* __restrict__ qw, int16_t* __restrict__ out, int64_t ntiles) {
  // thread = (tile, row pair q); the 8 threads of a tile are consecutive lanes
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const bool live = gid < ntiles * 8;
  StreamRegs<K> r;
#pragma unroll
  for (int k = 0; k < K; ++k) r.d[k] = 0u;
  if (live) load_stream<K>(qw + gid * K, r);
  const uint32_t prev = (uint32_t)__builtin_amdgcn_ds_bpermute(history_lane_byteaddr(lane), (int)r.d[K - 1]);
  if (!live) return;
  Window<K> w;
  w.build(r, prev);
  int16_t vals[32];
  ForEach32<K, 0>::run(w, [&](int u, int v) { vals[u] = (int16_t)v; });
  u4* o = (u4*)(out + gid * 32);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    u4 pk;
    pk.x = (uint16_t)vals[8 * i + 0] | ((uint32_t)(uint16_t)vals[8 * i + 1] << 16);
    pk.y = (uint16_t)vals[8 * i + 2] | ((uint32_t)(uint16_t)vals[8 * i + 3] << 16);
    pk.z = (uint16_t)vals[8 * i + 4] | ((uint32_t)(uint16_t)vals[8 * i + 5] << 16);
    pk.w = (uint16_t)vals[8 * i + 6] | ((uint32_t)(uint16_t)vals[8 * i + 7] << 16);
    o[i] = pk;
  }
}

template <int K>
__global__ __launch_bounds__(256) void k_dequant_q(const uint32_t* __restrict__ qw, const uint16_t* __restrict__ scales,
                                                   float* __restrict__ Q, int mt, int nt, double rms) {
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const int64_t ntiles = (int64_t)mt * nt;
  const bool live = gid < ntiles * 8;
  StreamRegs<K> r;
#pragma unroll
  for (int k = 0; k < K; ++k) r.d[k] = 0u;
  if (live) load_stream<K>(qw + gid * K, r);
  const uint32_t prev = (uint32_t)__builtin_amdgcn_ds_bpermute(history_lane_byteaddr(lane), (int)r.d[K - 1]);
  if (!live) return;
  Window<K> w;
  w.build(r, prev);
  const int64_t tile = gid >> 3;
  const int q = (int)(gid & 7);
  const int ti = (int)(tile / nt), tj = (int)(tile - (int64_t)ti * nt);
  const int64_t n = (int64_t)nt * 16;
  const int row0 = ti * 16 + 2 * q;
  const float sc0 = f16_bits_to_float(scales[row0]), sc1 = f16_bits_to_float(scales[row0 + 1]);
  float* o0 = Q + (int64_t)row0 * n + (int64_t)tj * 16;
  float* o1 = o0 + n;
  // cb[s] = float32(v / rms) with the division in float64, then one float32 multiply (htr/wire.py:24,102 of the reference)
  ForEach32<K, 0>::run(w, [&](int u, int v) {
    const float cb = (float)((double)v / rms);
    if (u < 16) o0[u] = cb * sc0; else o1[u - 16] = cb * sc1;
  });
}

// ------------------------------------------------------------------------------------------------ original-basis W
// W = Sv . Ho . Q . Hi . Su as bf16 [m, n] (htr/wire.py:105-113 of the reference), one workgroup of 512 threads per
// 128x128 block, 32 elements per thread.  Each H128 is seven butterfly stages, one per bit of the column or row index, and
// they commute:
//   matrix unit     column bits 0-4: wave w = (row half w % 2, column quarter w / 2) decodes 64 rows x 32 columns, and the decode
//                   registers are the A operands of v_mfma_f32_32x32x16_f16 as they are (see k_linear_tile); the B operand
//                   is H32, two constant fragments.  Whole numbers below 2^17: the products and sums are exact, and the
//                   1534 that every decoded half carries is removed by the accumulator's start value.
//   then registers  the row scale (times CBSCALE / 128, the two rotations' norms), row bits 0, 1, 2, 4, 5, which the matrix
//                   unit's output layout keeps inside a lane
//   LDS, registers  one trip re-deals the block: row bits 3 and 6, column bits 5 and 6; signs on the packed bf16 pairs.
// Bound: vector issue (about 3.3 decode instructions and 11 others per element), then the writes of W.  14336x4096 at K4: 45 -> 38.5 us
// against fourteen butterfly stages in registers with two trips through LDS.  (Workgroups that walk over several column blocks,
// the next block's words requested early, took 42 us: the start of a block is not what it waits for, and the grid fills worse.)
constexpr int DQW_LD = 132;   // LDS leading dimension in floats: 4 banks of shift per row, 32 per 8 rows
// position of a row in LDS: 16 rows further is another 32 banks, so that both half-waves' reads are free of conflicts
__device__ __forceinline__ int dqw_row(int row) { return row * DQW_LD + (row >> 4) * 32; }
constexpr size_t DQW_LDS = ((size_t)128 * DQW_LD + 7 * 32 + 128) * sizeof(float);      // the block, the row scales

// in-place Walsh-Hadamard butterflies over the index bits [B0, B1) of a 32-element register array
template <int B0, int B1> __device__ __forceinline__ void fwht_regs(float (&v)[32]) {
#pragma unroll
  for (int b = B0; b < B1; ++b)
#pragma unroll
    for (int i = 0; i < 32; ++i)
      if (!(i & (1 << b))) {
        const float x = v[i], y = v[i | (1 << b)];
        v[i] = x + y; v[i | (1 << b)] = x - y;
      }
}

typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float fl2 __attribute__((ext_vector_type(2)));

template <int K>
__global__ __launch_bounds__(512, 4) void k_dequant_w(const uint32_t* __restrict__ qw, const uint16_t* __restrict__ scales,
                                                      const uint8_t* __restrict__ su, const uint8_t* __restrict__ sv,
                                                      uint16_t* __restrict__ W, int nt, float cbscale) {
  extern __shared__ __align__(16) unsigned char lds[];
  float* blk = (float*)lds;                                  // rows at dqw_row()
  float* s_scale = blk + 128 * DQW_LD + 7 * 32;              // [128]
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int rh = w & 1, cq = w >> 1, l32 = lane & 31, kg = lane >> 5;
  const int bj = blockIdx.x, bi = blockIdx.y;                // 128-column block, 128-row block
  const int n = nt * 16;
  // ---- decode: lane = (tile column 2 cq + kg, strip 4 rh + l32 / 8, row pair lane % 8)
  StreamRegs<K> r;
  load_stream<K>(qw + ((size_t)(bi * 8 + 4 * rh + (l32 >> 3)) * nt + (size_t)bj * 8 + 2 * cq + kg) * (8 * K) + (lane & 7) * K, r);
  if (threadIdx.x < 128) s_scale[threadIdx.x] = f16_bits_to_float(scales[bi * 128 + threadIdx.x]) * cbscale * (1.0f / 128.0f);
  // H32: k-slot e of lane (column l32, k-group kg) stands for column 16 kg + 8 hf + e of the quarter
  h8 H[2];
#pragma unroll
  for (int hf = 0; hf < 2; ++hf)
#pragma unroll
    for (int e = 0; e < 8; ++e) H[hf][e] = (__builtin_popcount((16 * kg + 8 * hf + e) & l32) & 1) ? (_Float16)-1.f : (_Float16)1.f;
  DecodedStep<K> d;
  decode_step<K>(r, history_lane_byteaddr(lane), d);
  const float start = l32 == 0 ? -1534.f * 32.f : 0.f;       // the sum of H32's column is 32 for column 0, else 0
  f16v acc[2];
#pragma unroll
  for (int par = 0; par < 2; ++par) {
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[par][i] = start;
    acc[par] = __builtin_amdgcn_mfma_f32_32x32x16_f16(d.a[2 * par], H[0], acc[par], 0, 0, 0);
    acc[par] = __builtin_amdgcn_mfma_f32_32x32x16_f16(d.a[2 * par + 1], H[1], acc[par], 0, 0, 0);
  }
  __syncthreads();                                           // s_scale
  // register 4 rq + i of parity par is row 64 rh + 16 rq + 8 kg + 2 i + par, column 32 cq + l32 (as in k_linear_tile)
  float v[32];
#pragma unroll
  for (int rq = 0; rq < 4; ++rq) {
    const float* sp = s_scale + 64 * rh + 16 * rq + 8 * kg;
    const f4 lo = *(const f4*)sp, hi = *(const f4*)(sp + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[8 * rq + 2 * i] = acc[0][4 * rq + i] * (i < 2 ? lo[2 * i] : hi[2 * i - 4]);
      v[8 * rq + 2 * i + 1] = acc[1][4 * rq + i] * (i < 2 ? lo[2 * i + 1] : hi[2 * i - 3]);
    }
  }
  fwht_regs<0, 5>(v);                                        // row bits 0, 1, 2, 4, 5
  {
    float* p = blk + dqw_row(64 * rh) + 8 * kg * DQW_LD + 32 * cq + l32;
#pragma unroll
    for (int u = 0; u < 32; ++u) p[(u & 7) * DQW_LD + (u >> 3) * (16 * DQW_LD + 32)] = v[u];
  }
  // ---- second half: lane = columns 2 (lane % 16) + {0, 1}, row bits 4 and 0; wave = row bits 1, 2, 5;
  // v[c0 + 2 a0 + 4 a1 + 8 c] = row rbase + 8 a0 + 64 a1, column col + c0 + 32 c
  const int col = 2 * (lane & 15);
  const int rbase = 16 * ((lane >> 4) & 1) + (lane >> 5) + 2 * (w & 1) + 4 * ((w >> 1) & 1) + 32 * (w >> 2);
  uint32_t subits[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) subits[c] = (uint32_t)su[bj * 16 + 4 * c + (col >> 3)];
  const uint32_t* svw = (const uint32_t*)(sv + bi * 16);
  const uint32_t sv_lo = svw[w >> 2], sv_hi = svw[(w >> 2) + 2];      // rows rbase .., rbase + 64 ..
  __syncthreads();
  const float* p = blk + dqw_row(rbase) + col;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const fl2 t = *(const fl2*)(p + (i & 1) * (8 * DQW_LD) + ((i >> 1) & 1) * (64 * DQW_LD + 4 * 32) + 32 * (i >> 2));
    v[2 * i] = t.x; v[2 * i + 1] = t.y;
  }
  fwht_regs<1, 5>(v);                                        // row bits 3, 6, column bits 5, 6
  uint16_t* dst = W + (size_t)(bi * 128 + rbase) * n + (size_t)bj * 128 + col;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const uint32_t sbit = (((a >> 1) ? sv_hi : sv_lo) >> ((rbase & 31) + 8 * (a & 1))) & 1u;      // rbase & 31 has bit 3 clear
    const uint32_t rowmask = sbit * 0x80008000u;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t sb = subits[c] >> (col & 7);
      const fl2 f = {v[2 * a + 8 * c], v[2 * a + 8 * c + 1]};
      const bf2 h = __builtin_convertvector(f, bf2);
      *(uint32_t*)(dst + (size_t)(8 * (a & 1) + 64 * (a >> 1)) * n + 32 * c) =
          __builtin_bit_cast(uint32_t, h) ^ ((sb & 1u) << 15) ^ ((sb & 2u) << 30) ^ rowmask;
    }
  }
}
