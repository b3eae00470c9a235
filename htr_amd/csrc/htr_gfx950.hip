// HTR-W1 packed-linear kernels for MI355X (gfx950, CDNA4, wave64) behind a plain C ABI.
//
//   y = sv . Ho( Q . Hi(su . x) ),   Q[i,j] = v(s_ij) * scale_i * CBSCALE,
//   v(s) = bytesum((s * 0xDF6ADF + 0x34983) mod 2^32) - 510              (docs/FORMAT.md:7-13 of the reference)
//
// Work decomposition of the fused linear kernel
//   step      = one 128-row x 128-column block of the weight; the steps of a linear, row-major, are cut into equal
//               contiguous chunks, one workgroup each, so the workgroup count does not depend on the shape
//   workgroup = 8 waves = the 8 strips of a 128-row block (one H128 output block)
//   wave      = one 16-row strip of tiles; per step it streams the 8 consecutive tiles that cover one 128-column
//               input block (8 * 32K contiguous bytes: each lane loads its 4K contiguous bytes) through a buffer
//               descriptor that covers exactly its bytes of the chunk, so loads beyond the end cost nothing
//   lane      = (tile-in-step = lane / 8, row pair q = lane % 8): the K dwords a lane loads are exactly the stream
//               bits of tile rows 2q and 2q+1 (32 steps); the 16-K history bits come from the previous lane's last
//               dword through the LDS crossbar (ds_bpermute), the tail-biting wrap is lane 7 -> lane 0 of the tile
//   decode    = per weight: one bit-field extract, one v_mad_u32_u24, one v_sad_u8 / v_sad_hi_u8.  The SAD pair
//               accumulates onto 0x64006400, which leaves two IEEE half floats 1024 + bytesum = 1534 + v packed in
//               one dword with no integer->float conversion and no pack instruction.
//   product   = v_mfma_f32_16x16x32_f16.  MFMA row i = lane % 16 = (tile parity h = i / 8, row pair q = i % 8), the
//               four 16-lane groups g supply the k-slots, so lane (g, h, q) feeds tile 2g + h.  Rows with h = 0 and
//               h = 1 need different activation columns; the B operand therefore carries, for activation row r,
//               the even tiles in MFMA column 2r and the odd tiles in column 2r + 1, and only D[i][2r + h(i)] is
//               kept.  Eight activation rows share one MFMA; more rows reuse the decoded A registers.
//   offset    = the constant 1534 is removed afterwards with 1534 * sum(x~) per activation row.
//   epilogue  = the workgroup whose chunk holds the last step of a row block finishes it: it adds the partials the
//               earlier chunks of that row block left in their workspace slots (fixed order) to its own, applies
//               scale * CBSCALE, the output H128, sv, bias and the cast.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>
#include <stdlib.h>
#include <atomic>
#include <mutex>
#include <type_traits>

#include "../../include/htr_gfx950.h"

namespace {
#include "decode.hpp"
#include "linear.hpp"
#include "linear_batch.hpp"
#include "linear_tile.hpp"
#include "linear_gemm.hpp"
#include "linear_wide.hpp"
#include "moe.hpp"
#include "dequant.hpp"
#include "viterbi.hpp"
#include "anchors.hpp"
#include "plan.hpp"
}  // namespace

// ================================================================================================ C ABI
extern "C" {

const char* htr_strerror(int status) {
  switch (status) {
    case HTR_OK: return "ok";
    case HTR_ERR_NULL: return "a required pointer is NULL";
    case HTR_ERR_K: return "unsupported K (HTR-W1 allows 2..8)";
    case HTR_ERR_SHAPE: return "m and n must be positive multiples of 128";
    case HTR_ERR_BATCH: return "M must be in 1..2048 for one launch (1..128 for an explicit chunked or batched plan, 1..32 for a grouped problem)";
    case HTR_ERR_DTYPE: return "dtype must be bf16 (0), f16 (1) or f32 (2)";
    case HTR_ERR_WORKSPACE: return "workspace too small or not 256-byte aligned";
    case HTR_ERR_ALIGN: return "tensor pointer not aligned (qweight 16 B, others natural)";
    case HTR_ERR_LAUNCH: return "HIP launch failed";
    case HTR_ERR_SPLIT: return "explicit split count does not fit this shape";
    case HTR_ERR_COUNT: return "problem count out of range";
    default: return "unknown status";
  }
}

int htr_last_hip_error(void) { return g_last_hip_error; }
int htr_abi_version(void) { return HTR_ABI_VERSION; }
float htr_cbscale(void) { return (float)(1.0 / __builtin_sqrt(MEAN_SQ)); }

size_t htr_workspace_bytes(int m, int n, int K, int M, int nsplit) {
  if (K < 2 || K > 8 || !shape_ok(m, n) || M < 1 || M > HTR_MAX_BATCH) return 0;
  if (wants_wide(M, nsplit)) {
    WidePlan wp;
    if (!make_wide_plan(m, n, M, wide_want_S(nsplit), wp)) return 0;
    // up to 128 rows a slot per workgroup whatever the plan, as the batched kernel's plans: a workspace for one serves the other
    const size_t slots = nsplit > 0 ? wide_slot_bytes(m, M, wp) : (size_t)wp.wgs * M * 128 * sizeof(float);
    return ws_need(slots, prerot_bytes(n, M));
  }
  if (wants_gemm(M, nsplit)) {
    GemmPlan gp;
    if (!make_gemm_plan(m, n, M, nsplit > 0 ? nsplit & 0xFFFFF : 0, gemm_want_jb(nsplit), gp)) return 0;
    return ws_need((size_t)gp.wgs * sizeof(uint32_t), gemm_scratch_bytes(n, M, gp));
  }
  if (M > HTR_MAX_ROWS_PER_TILE) return 0;       // the other kernels take up to 128 rows
  if (wants_batch(M, nsplit, m, n, K)) {
    BatchPlan bp;
    if (!make_batch_plan(m, n, K, M, nsplit > 0 ? nsplit & 0xFFFFF : 0, bp)) return 0;
    return ws_need((size_t)bp.wgs * M * 128 * sizeof(float), prerot_bytes(n, batch_prerot_rows(M, bp.tile)));
  }
  if (M > HTR_MAX_GROUP_ROWS) return 0;          // the chunked kernel takes up to 32 rows
  Plan pl;
  if (!make_plan(m, n, K, M, nsplit, pl)) return 0;
  return ws_need((size_t)pl.wgs * M * 128 * sizeof(float), prerot_bytes(n, M));
}

// the chunked kernel's own rotation reads 16-bit elements in pairs: float32 activations, and rows that do not start on a
// 4-byte boundary, take the pre-rotation
static bool chunks_prerotated(const Plan& pl, int x_dtype, const void* x) { return pl.prerot || x_dtype == HTR_F32 || ((uintptr_t)x & 3); }

int htr_linear_rotation(int m, int n, int K, int M, int nsplit, int x_dtype, const void* x) {
  int out6[6];
  const int rc = htr_linear_plan(m, n, K, M, nsplit, out6);
  if (rc != HTR_OK) return -rc;
  if (!dtype_ok(x_dtype)) return -HTR_ERR_DTYPE;
  if ((uintptr_t)x & (x_dtype == HTR_F32 ? 3 : 1)) return -HTR_ERR_ALIGN;
  if (wants_wide(M, nsplit) || wants_gemm(M, nsplit)) return 0;
  BatchPlan bp;
  if (wants_batch(M, nsplit, m, n, K)) return make_batch_plan(m, n, K, M, nsplit > 0 ? nsplit & 0xFFFFF : 0, bp) ? batch_rot(K, M, x_dtype, x, bp) : -HTR_ERR_SPLIT;
  Plan pl;
  return make_plan(m, n, K, M, nsplit, pl) ? !chunks_prerotated(pl, x_dtype, x) : -HTR_ERR_SPLIT;
}

int htr_linear_plan(int m, int n, int K, int M, int nsplit, int* out6) {
  if (!out6) return HTR_ERR_NULL;
  if (K < 2 || K > 8) return HTR_ERR_K;
  if (!shape_ok(m, n)) return HTR_ERR_SHAPE;
  if (M < 1 || M > HTR_MAX_BATCH) return HTR_ERR_BATCH;
  if (wants_wide(M, nsplit)) {
    WidePlan wp;
    if (!make_wide_plan(m, n, M, wide_want_S(nsplit), wp)) return HTR_ERR_SPLIT;
    out6[0] = wp.cb; out6[1] = wp.wgs; out6[2] = nsplit > 0 ? wp.mtiles : (wp.wgs > num_cu() ? 0 : 1); out6[3] = wp.S; out6[4] = 1; out6[5] = (int)WIDE_LDS;
    return HTR_OK;
  }
  if (wants_gemm(M, nsplit)) {
    GemmPlan gp;
    if (!make_gemm_plan(m, n, M, nsplit > 0 ? nsplit & 0xFFFFF : 0, gemm_want_jb(nsplit), gp)) return HTR_ERR_SPLIT;
    out6[0] = gp.cb; out6[1] = gp.wgs; out6[2] = gp.mtiles; out6[3] = gp.S; out6[4] = 1; out6[5] = (int)gemm_lds_bytes(gp.jb);
    return HTR_OK;
  }
  if (M > HTR_MAX_ROWS_PER_TILE) return HTR_ERR_BATCH;
  if (wants_batch(M, nsplit, m, n, K)) {
    BatchPlan bp;
    if (!make_batch_plan(m, n, K, M, nsplit > 0 ? nsplit & 0xFFFFF : 0, bp)) return HTR_ERR_SPLIT;
    out6[0] = bp.cb; out6[1] = bp.wgs; out6[2] = bp.last_finishes ? 0 : 1; out6[3] = bp.S; out6[4] = bp.rot ? 0 : 1; out6[5] = (int)bp.lds;
    return HTR_OK;
  }
  if (M > HTR_MAX_GROUP_ROWS) return HTR_ERR_BATCH;
  Plan pl;
  if (!make_plan(m, n, K, M, nsplit, pl)) return HTR_ERR_SPLIT;
  out6[0] = pl.chunk; out6[1] = pl.wgs; out6[2] = pl.segfin; out6[3] = pl.nbl; out6[4] = pl.prerot; out6[5] = (int)pl.lds;
  return HTR_OK;
}

int htr_linear_route(int m, int n, int K, int M, int x_dtype, int eager) {
  const int refused = K < 2 || K > 8 ? HTR_ERR_K : !shape_ok(m, n) ? HTR_ERR_SHAPE : M < 1 || M > HTR_MAX_BATCH ? HTR_ERR_BATCH : !dtype_ok(x_dtype) ? HTR_ERR_DTYPE : HTR_OK;
  if (refused != HTR_OK) return HTR_ROUTE_DEQUANTIZE - refused;
  if (M <= HTR_MAX_ROWS_PER_TILE) return 0;
  WidePlan wp;
  const bool wide = make_wide_plan(m, n, M, 0, wp);
  if (M <= fused_rows(m, n)) return wide ? NSPLIT_WIDE : 0;
  return wide && x_dtype != HTR_F32 && wide_ahead(m, n, K, M, x_dtype, wp, eager != 0) ? NSPLIT_WIDE : HTR_ROUTE_DEQUANTIZE;
}

void htr_set_spin_limit(int polls) { g_spin_limit.store(polls < 1 ? 1 : polls, std::memory_order_relaxed); }

int htr_plan_device_override(int compute_units, long lds_bytes_per_cu) {
  if (compute_units == 0) { g_override_cus.store(0, std::memory_order_release); return HTR_OK; }
  if (compute_units < 1 || compute_units > 4096 || lds_bytes_per_cu < 64 * 1024 || lds_bytes_per_cu > (1 << 20)) return HTR_ERR_SHAPE;
  g_override_lds.store(lds_bytes_per_cu, std::memory_order_release);
  g_override_cus.store(compute_units, std::memory_order_release);
  return HTR_OK;
}

int htr_workspace_init(void* workspace, size_t workspace_bytes, void* host_status_word, void* stream) {
  if (!workspace) return HTR_ERR_NULL;
  if (workspace_bytes < 2 * WS_HEADER || ((uintptr_t)workspace & 255) || ((uintptr_t)host_status_word & 3)) return HTR_ERR_WORKSPACE;
  const size_t half = ws_half(workspace_bytes);
  const size_t n16 = half / 16;
  const unsigned blocks = (unsigned)(n16 / 256 < 1 ? 1 : (n16 / 256 > 2048 ? 2048 : n16 / 256));
  HTR_CHECK_HIP(launch_kernel(k_workspace_init, dim3(blocks), dim3(256), 0, (hipStream_t)stream, (u4*)workspace, half,
                              (unsigned long long)(uintptr_t)host_status_word));
  return HTR_OK;
}

namespace {
// The launches of one call on a workspace stay together in their stream: two host threads that share a stream, and with it a
// workspace, would otherwise rotate into the scratch half that the other one's product is about to read.  One of 64 locks by
// address, held while the launches are queued.
struct Together {
  std::mutex& m;
  static std::mutex& of(const void* workspace) {
    static std::mutex locks[64];
    return locks[((uint64_t)(uintptr_t)workspace >> 8) * 0x9E3779B97F4A7C15ull >> 58];
  }
  explicit Together(const void* workspace) : m(of(workspace)) { m.lock(); }
  ~Together() { m.unlock(); }
  Together(const Together&) = delete;
};
}

unsigned long long htr_stream_capture_id(void* stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo((hipStream_t)stream, &status, &id) != hipSuccess) { (void)hipGetLastError(); return 0; }
  return status == hipStreamCaptureStatusActive ? (id != 0 ? id : ~0ull) : 0;
}

int htr_linear(const void* qweight, const void* scales, const void* su, const void* sv, const void* x, const void* bias,
               void* y, int m, int n, int K, int M, int x_dtype, int y_dtype, int nsplit, void* workspace,
               size_t workspace_bytes, void* stream) {
  if (!qweight || !scales || !su || !sv || !x || !y) return HTR_ERR_NULL;
  if (K < 2 || K > 8) return HTR_ERR_K;
  if (!shape_ok(m, n)) return HTR_ERR_SHAPE;
  if (M < 1 || M > HTR_MAX_BATCH) return HTR_ERR_BATCH;
  if (!dtype_ok(x_dtype) || !dtype_ok(y_dtype)) return HTR_ERR_DTYPE;
  if (((uintptr_t)qweight & 15) || ((uintptr_t)scales & 1) || ((uintptr_t)x & (x_dtype == HTR_F32 ? 3 : 1)) ||
      ((uintptr_t)y & (y_dtype == HTR_F32 ? 3 : 1)) || (bias && ((uintptr_t)bias & (y_dtype == HTR_F32 ? 3 : 1))))
    return HTR_ERR_ALIGN;
  const Together together(workspace);
  if (wants_wide(M, nsplit)) {
    WidePlan wp;
    if (!make_wide_plan(m, n, M, wide_want_S(nsplit), wp)) return HTR_ERR_SPLIT;
    const size_t need = htr_workspace_bytes(m, n, K, M, nsplit);
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255)) return HTR_ERR_WORKSPACE;
    LinearTail t = {};
    t.scales = (const uint16_t*)scales; t.sv = (const uint8_t*)sv; t.bias = bias; t.y = y;
    place_prerot(t, (unsigned char*)workspace + ws_half(workspace_bytes), n, M);
    t.status = (uint32_t*)workspace;
    t.cbscale = htr_cbscale();
    t.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
    hipStream_t st = (hipStream_t)stream;
    HTR_CHECK_HIP(launch_rotation(x, (const uint8_t*)su, n, M, x_dtype, t, st, (size_t)M));
    const BatchArgs a = {(const uint32_t*)qweight, (float*)((unsigned char*)workspace + WS_HEADER), nullptr, nullptr, m, n, M,
                         x_dtype | (y_dtype << 2) | (wp.wgs > num_cu() ? FLAG_LAST_FINISHES : 0)};
    HTR_FOR_K(K, return launch_wide_k<KK>(a, t, wp, st));
    return HTR_OK;
  }
  if (wants_gemm(M, nsplit)) {
    GemmPlan gp;
    if (!make_gemm_plan(m, n, M, nsplit > 0 ? nsplit & 0xFFFFF : 0, gemm_want_jb(nsplit), gp)) return HTR_ERR_SPLIT;
    const size_t need = htr_workspace_bytes(m, n, K, M, nsplit);
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255)) return HTR_ERR_WORKSPACE;
    unsigned char* wsp = (unsigned char*)workspace + ws_half(workspace_bytes);
    LinearTail t;
    t.scales = (const uint16_t*)scales; t.sv = (const uint8_t*)sv; t.bias = bias; t.y = y;
    t.xt_g = (const _Float16*)wsp;
    t.xs_g = (const float*)(wsp + align256((size_t)M * n * 2));
    t.sc_g = (const float*)(wsp + align256((size_t)M * n * 2) + align256((size_t)M * (n / 128) * 16));
    t.tiles = (float*)(wsp + prerot_bytes(n, M));
    t.status = (uint32_t*)workspace;
    t.cbscale = htr_cbscale();
    t.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
    t.chunk_magic = 0;
    t.group = nullptr; t.group_prerot_stride = 0; t.group_part_stride = 0;
    hipStream_t st = (hipStream_t)stream;
    HTR_CHECK_HIP(launch_rotation(x, (const uint8_t*)su, n, M, x_dtype, t, st));
    const uint32_t* qwp = (const uint32_t*)qweight;
    float* flags = (float*)((unsigned char*)workspace + WS_HEADER);
    const int flg = x_dtype | (y_dtype << 2);
#define HTR_LAUNCH_GEMM(KK_, PP_)                                                                                          \
    {                                                                                                                      \
      if (gp.jb == 3) {                                                                                                    \
        HTR_CHECK_HIP((allow_full_lds<k_linear_gemm<KK_, PP_, 3>>()));                                                     \
        HTR_CHECK_HIP(launch_kernel(k_linear_gemm<KK_, PP_, 3>, dim3(gp.S, m / 128, gp.mtiles), dim3(GEMM_THREADS),        \
                                    gemm_lds_bytes(3), st, qwp, flags, m, n, M, gp.S, flg, t));                            \
      } else {                                                                                                             \
        HTR_CHECK_HIP((allow_full_lds<k_linear_gemm<KK_, 2, 4>>()));                                                       \
        HTR_CHECK_HIP(launch_kernel(k_linear_gemm<KK_, 2, 4>, dim3(gp.S, m / 128, gp.mtiles), dim3(GEMM_THREADS),          \
                                    gemm_lds_bytes(4), st, qwp, flags, m, n, M, gp.S, flg, t));                            \
      }                                                                                                                    \
    }
    switch (K) {
      case 2: HTR_LAUNCH_GEMM(2, 4); break;
      case 3: HTR_LAUNCH_GEMM(3, 4); break;
      case 4: HTR_LAUNCH_GEMM(4, 4); break;
      case 5: HTR_LAUNCH_GEMM(5, 2); break;
      case 6: HTR_LAUNCH_GEMM(6, 2); break;
      case 7: HTR_LAUNCH_GEMM(7, 2); break;
      default: HTR_LAUNCH_GEMM(8, 2); break;
    }
#undef HTR_LAUNCH_GEMM
    return HTR_OK;
  }
  if (M > HTR_MAX_ROWS_PER_TILE) return HTR_ERR_BATCH;        // explicit plans of the other kernels take up to 128 rows
  if (wants_batch(M, nsplit, m, n, K)) {
    BatchPlan bp;
    if (!make_batch_plan(m, n, K, M, nsplit > 0 ? nsplit & 0xFFFFF : 0, bp)) return HTR_ERR_SPLIT;
    const size_t need = htr_workspace_bytes(m, n, K, M, nsplit);
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255)) return HTR_ERR_WORKSPACE;
    unsigned char* wsp = (unsigned char*)workspace + ws_half(workspace_bytes);
    LinearTail t;
    t.scales = (const uint16_t*)scales; t.sv = (const uint8_t*)sv; t.bias = bias; t.y = y;
    place_prerot(t, wsp, n, batch_prerot_rows(M, bp.tile));
    t.status = (uint32_t*)workspace;
    t.cbscale = htr_cbscale();
    t.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
    t.chunk_magic = 0;
    t.group = nullptr; t.group_prerot_stride = 0; t.group_part_stride = 0; t.tiles = nullptr;
    hipStream_t st = (hipStream_t)stream;
    const int rot = batch_rot(K, M, x_dtype, x, bp);
    if (!rot) HTR_CHECK_HIP(launch_rotation(x, (const uint8_t*)su, n, M, x_dtype, t, st, bp.tile ? FRAG_FULL : 0));
    BatchArgs ba;
    ba.qw = (const uint32_t*)qweight; ba.part = (float*)((unsigned char*)workspace + WS_HEADER); ba.x = x; ba.su = (const uint8_t*)su;
    ba.m = m; ba.n = n; ba.M = M; ba.flags = x_dtype | (y_dtype << 2) | (bp.last_finishes ? FLAG_LAST_FINISHES : 0);
    bp.lds = rot ? batch_rot_lds_bytes(M, bp.cb, rot) : batch_lds_bytes(M, bp.tile);
    HTR_FOR_K(K, return launch_batch_k<KK>(ba, rot, t, bp, st));
    return HTR_OK;
  }
  if (M > HTR_MAX_GROUP_ROWS) return HTR_ERR_BATCH;          // an explicit chunked plan: that kernel takes up to 32 rows
  Plan pl;
  if (!make_plan(m, n, K, M, nsplit, pl)) return HTR_ERR_SPLIT;
  const bool prerot = chunks_prerotated(pl, x_dtype, x);
  const size_t need = htr_workspace_bytes(m, n, K, M, nsplit);
  if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255)) return HTR_ERR_WORKSPACE;

  unsigned char* wsp = (unsigned char*)workspace + ws_half(workspace_bytes);      // scratch half
  LinearLaunch a;
  a.qw = (const uint32_t*)qweight; a.x = x; a.su = (const uint8_t*)su;
  a.part = (float*)((unsigned char*)workspace + WS_HEADER);
  a.m = m; a.n = n; a.M = M; a.chunk = pl.chunk; a.flags = x_dtype | (y_dtype << 2); a.problems = 1;
  // Eight lanes of whole row blocks, one per XCD: possible when the chunks tile the rows of column blocks and the row
  // blocks divide by eight.  Measured on MI355X (K4, batch 1): -0.2 us on 4096x4096, -0.3 us on 4096x14336 (eight chunks
  // per row block), no change with two chunks per row block, +0.1 us with a single row block per lane (1024x4096),
  // hence the lower bound of two row blocks per lane.  HTR_LANES=0 switches it off.
  {
    static const bool lanes_on = getenv("HTR_LANES") == nullptr || atoi(getenv("HTR_LANES")) != 0;
    const int nblk = n / 128, rbs = m / 128;
    if (lanes_on && pl.chunk < nblk && nblk % pl.chunk == 0 && rbs % 8 == 0 && rbs >= 16 && pl.wgs % 8 == 0) a.flags |= FLAG_LANES | ((pl.wgs / 8) << FLAG_LANE_LEN_SHIFT);
  }
  a.nblk_magic = (((unsigned long long)1 << 40) + (unsigned)(n / 128) - 1) / (unsigned)(n / 128);
  LinearTail& t = a.tail;
  t.scales = (const uint16_t*)scales; t.sv = (const uint8_t*)sv; t.bias = bias; t.y = y;
  t.xt_g = nullptr; t.xs_g = nullptr; t.sc_g = nullptr;
  t.status = (uint32_t*)workspace;
  t.cbscale = htr_cbscale();
  t.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
  t.group = nullptr; t.group_prerot_stride = 0; t.group_part_stride = 0; t.tiles = nullptr;
  t.chunk_magic = (((unsigned long long)1 << 40) + (unsigned)pl.chunk - 1) / (unsigned)pl.chunk;
  hipStream_t st = (hipStream_t)stream;
  if (prerot) {
    t.xt_g = (const _Float16*)wsp;
    t.xs_g = (const float*)(wsp + align256((size_t)M * n * 2));
    t.sc_g = (const float*)(wsp + align256((size_t)M * n * 2) + align256((size_t)M * (n / 128) * 16));
    HTR_CHECK_HIP(launch_rotation(x, (const uint8_t*)su, n, M, x_dtype, t, st));
  }
  HTR_FOR_K(K, return launch_linear_k<KK>(a, prerot, pl.mb, pl.wgs, pl.lds, st));
  return HTR_OK;
}

// ---- htr_linear for callers that can neither allocate nor bring a workspace: the workspace is an array in the
// library's own device image.  Host code only ever holds the address hipGetSymbolAddress returns for it on the current
// device (every device has its own copy of the array at its own address; the symbol's name itself is no device address).
static __device__ __align__(256) unsigned char scratch[HTR_STATIC_SCRATCH_BYTES];

namespace {
void* g_scratch_ptr[MAX_DEVICES];                 // per device: address of `scratch` there, once looked up
std::atomic<uint64_t> g_scratch_known{0};         // bit d: g_scratch_ptr[d] is valid
}

int htr_linear_static(const void* qweight, const void* scales, const void* su, const void* sv, const void* x, const void* bias,
                      void* y, int m, int n, int K, int M, int x_dtype, int y_dtype, int reset, void* stream) {
  if (K < 2 || K > 8) return HTR_ERR_K;
  if (!shape_ok(m, n)) return HTR_ERR_SHAPE;
  if (M < 1 || M > HTR_MAX_BATCH) return HTR_ERR_BATCH;
  const size_t need = htr_workspace_bytes(m, n, K, M, 0);
  if (need == 0 || need > (size_t)HTR_STATIC_SCRATCH_BYTES) return HTR_ERR_WORKSPACE;      // beyond the built-in workspace
  int dev = 0;
  HTR_CHECK_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= MAX_DEVICES) { g_last_hip_error = (int)hipErrorInvalidDevice; return HTR_ERR_LAUNCH; }
  const uint64_t bit = (uint64_t)1 << dev;
  if (!(g_scratch_known.load(std::memory_order_acquire) & bit)) {
    void* p = nullptr;
    HTR_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev] = p;                       // two threads racing here store the same address
    g_scratch_known.fetch_or(bit, std::memory_order_release);
  }
  void* ws = g_scratch_ptr[dev];
  if (reset) {
    const int rc = htr_workspace_init(ws, HTR_STATIC_SCRATCH_BYTES, nullptr, stream);
    if (rc != HTR_OK) return rc;
  }
  return htr_linear(qweight, scales, su, sv, x, bias, y, m, n, K, M, x_dtype, y_dtype, 0, ws, HTR_STATIC_SCRATCH_BYTES, stream);
}

// plan of a grouped launch: every problem has the same shape, so one plan serves all; the activations are always
// rotated ahead (one launch for all problems) and the chunk is chosen for the whole grid
static bool make_group_plan(int count, int m, int n, int max_M, Plan& pl) {
  const int nblk = n / 128, rbs = m / 128;
  const long vtotal = (long)rbs * nblk;
  pl.mb = max_M <= 8 ? 1 : 2;      // up to 12 rows come here (group_takes_tiles)
  // aim at a few workgroups per CU over all problems; chunks are whole rows of column blocks or divide one, so that
  // no chunk straddles a row block; of those the one nearest the target (in ratio) that fits LDS
  static const int per_cu = getenv("HTR_GROUP_WGS_PER_CU") ? atoi(getenv("HTR_GROUP_WGS_PER_CU")) : 4;
  const double target = (double)vtotal * count / ((double)(per_cu > 0 ? per_cu : 4) * num_cu());
  double best = 1e30;
  bool found = false;
  for (long chunk = 1; chunk <= vtotal && chunk <= MAX_CHUNK; ++chunk) {
    if (chunk < nblk ? nblk % chunk != 0 : chunk % nblk != 0) continue;
    Plan c;
    c.mb = pl.mb;
    if (!plan_for_chunk(m, n, max_M, (int)chunk, c)) continue;
    const double ratio = chunk > target ? chunk / target : target / chunk;
    if (ratio < best) { best = ratio; pl = c; found = true; }
  }
  pl.prerot = 1;
  return found;
}

size_t htr_grouped_workspace_bytes(int count, int m, int n, int K, int max_M) {
  if (K < 2 || K > 8 || !shape_ok(m, n) || max_M < 1 || max_M > HTR_MAX_GROUP_ROWS || count < 1 || count > HTR_MAX_GROUP) return 0;
  if (group_takes_tiles(count, m, n, K, max_M)) {                 // one row tile per problem, partials only with column splits
    const int S = group_tile_splits(count, m, n);
    return ws_need(S > 1 ? (size_t)count * (m / 128) * S * max_M * 128 * sizeof(float) : 0, prerot_bytes(n, (size_t)32 * count));
  }
  Plan pl;
  if (!make_group_plan(count, m, n, max_M, pl)) return 0;
  return ws_need((size_t)count * pl.wgs * max_M * 128 * sizeof(float), (size_t)count * prerot_bytes(n, max_M));
}

int htr_linear_grouped(const htr_group_entry* entries, int count, int m, int n, int K, int max_M, int x_dtype, int y_dtype,
                       void* workspace, size_t workspace_bytes, void* stream) {
  if (!entries) return HTR_ERR_NULL;
  if (count < 1 || count > HTR_MAX_GROUP) return HTR_ERR_COUNT;
  if (K < 2 || K > 8) return HTR_ERR_K;
  if (!shape_ok(m, n)) return HTR_ERR_SHAPE;
  if (max_M < 1 || max_M > HTR_MAX_GROUP_ROWS) return HTR_ERR_BATCH;
  if (!dtype_ok(x_dtype) || !dtype_ok(y_dtype)) return HTR_ERR_DTYPE;
  if ((uintptr_t)entries & 7) return HTR_ERR_ALIGN;
  const size_t need = htr_grouped_workspace_bytes(count, m, n, K, max_M);
  if (need == 0) return HTR_ERR_SPLIT;
  if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255)) return HTR_ERR_WORKSPACE;

  const Together together(workspace);
  unsigned char* wsp = (unsigned char*)workspace + ws_half(workspace_bytes);      // scratch half
  if (group_takes_tiles(count, m, n, K, max_M)) {
    // one tile of 32 rows per problem
    LinearTail t = {};
    place_prerot(t, wsp, n, (size_t)32 * count);
    t.status = (uint32_t*)workspace;
    t.cbscale = htr_cbscale();
    t.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
    t.group = entries;
    hipStream_t st = (hipStream_t)stream;
    const int S = group_tile_splits(count, m, n);
    HTR_CHECK_HIP(launch_kernel(k_rotate, dim3((n / 128 + WG_WAVES - 1) / WG_WAVES, max_M, count), dim3(WG_THREADS), 0, st, (const void*)nullptr,
                                (const uint8_t*)nullptr, n, x_dtype, (_Float16*)t.xt_g, (float*)t.xs_g, (float*)t.sc_g, entries, 0ull, FRAG_FULL));
    BatchArgs ba = {nullptr, (float*)((unsigned char*)workspace + WS_HEADER), nullptr, nullptr, m, n, max_M, x_dtype | (y_dtype << 2)};
    HTR_FOR_K(K, return (S > 1 ? launch_tile_v<KK, 1, false>(ba, t, S, count, st) : launch_tile_v<KK, 1, true>(ba, t, 1, count, st)));
  }
  Plan pl;
  if (!make_group_plan(count, m, n, max_M, pl)) return HTR_ERR_SPLIT;
  const size_t pre = prerot_bytes(n, max_M);
  LinearLaunch a;
  a.qw = nullptr; a.x = nullptr; a.su = nullptr;
  a.part = (float*)((unsigned char*)workspace + WS_HEADER);
  a.m = m; a.n = n; a.M = max_M; a.chunk = pl.chunk; a.flags = x_dtype | (y_dtype << 2); a.problems = count;
  a.nblk_magic = (((unsigned long long)1 << 40) + (unsigned)(n / 128) - 1) / (unsigned)(n / 128);
  LinearTail& t = a.tail;
  t.scales = nullptr; t.sv = nullptr; t.bias = nullptr; t.y = nullptr;
  t.xt_g = (const _Float16*)wsp;
  t.xs_g = (const float*)(wsp + align256((size_t)max_M * n * 2));
  t.sc_g = (const float*)(wsp + align256((size_t)max_M * n * 2) + align256((size_t)max_M * (n / 128) * 16));
  t.status = (uint32_t*)workspace;
  t.cbscale = htr_cbscale();
  t.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
  t.chunk_magic = (((unsigned long long)1 << 40) + (unsigned)pl.chunk - 1) / (unsigned)pl.chunk;
  t.tiles = nullptr;
  t.group = entries; t.group_prerot_stride = pre; t.group_part_stride = (unsigned long long)pl.wgs * max_M * 128;
  hipStream_t st = (hipStream_t)stream;
  HTR_CHECK_HIP(launch_kernel(k_rotate, dim3((n / 128 + WG_WAVES - 1) / WG_WAVES, max_M, count), dim3(WG_THREADS), 0, st, (const void*)nullptr,
                              (const uint8_t*)nullptr, n, x_dtype, (_Float16*)t.xt_g, (float*)t.xs_g, (float*)t.sc_g, entries,
                              (unsigned long long)pre, (size_t)0));
  HTR_FOR_K(K, return launch_linear_k<KK>(a, true, pl.mb, pl.wgs, pl.lds, st));
  return HTR_OK;
}

// ---- routed experts: one MoE layer in a few launches (moe.hpp)
namespace {
struct MoePlan { int pairs, entries, tiles, rows; size_t table, e1, e2, pos, info, xt1, xs1, sc1, xt2, xs2, sc2, h, out, total; };
// Rows per table entry.  An entry decodes its expert's weights once, so few tall entries decode least; but a step of a tall tile
// takes longer also where it is half empty.  us of the layer with entries of 32 / 64 rows, by the mean rows of an expert: 64 experts,
// top 6, 2048x1408 K4: 15 rows 122 / 133, 18 rows 122 / 135, 24 rows 134 / 141, 28 rows 145 / 144, 31 rows 162 / 150, 46 rows
// 219 / 177; 8 experts, top 2, 4096x2048 K4: 16 rows 57 / 62, 24 rows 59 / 63, 32 rows 78 / 66; 16 experts, top 4, 1024x4096 K5:
// 18 rows 80 / 85, 25 rows 82 / 87, 32 rows 95 / 92.
inline int moe_rows_per_entry(int pairs, int experts) {
  const int active = experts < pairs ? experts : pairs;
  const int mean = pairs / active;
  return mean <= 25 ? 32 : 64;
}
inline bool moe_plan(int tokens, int top, int experts, int hidden, int inter, MoePlan& p) {
  if (tokens < 1 || top < 1 || experts < 1 || experts > MOE_MAX_EXPERTS || (long)tokens * top >= (1L << 24)) return false;
  if (!shape_ok(2 * inter, hidden) || !shape_ok(hidden, inter)) return false;
  p.pairs = tokens * top;
  p.rows = moe_rows_per_entry(p.pairs, experts);
  const int active = experts < p.pairs ? experts : p.pairs;
  p.entries = active + p.pairs / p.rows;
  p.tiles = active + p.pairs / 32;
  // with shape_ok and the pairs, every launch of the layer is within the grid's limits (65535 in y and z, 2^32 threads in x)
  if (p.entries > 65535) return false;
  size_t o = 0;
  auto take = [&](size_t bytes) { const size_t at = o; o += align256(bytes); return at; };
  p.table = take((size_t)experts * 64);
  p.e1 = take((size_t)p.entries * sizeof(htr_group_entry));
  p.e2 = take((size_t)p.entries * sizeof(htr_group_entry));
  p.pos = take((size_t)p.pairs * 4);
  p.info = take((size_t)p.pairs * 16);
  const size_t rows = (size_t)p.tiles * 32;
  p.xt1 = take(rows * hidden * 2); p.xs1 = take(rows * (hidden / 128) * 16); p.sc1 = take(rows * 4);
  p.xt2 = take(rows * inter * 2); p.xs2 = take(rows * (inter / 128) * 16); p.sc2 = take(rows * 4);
  p.h = take((size_t)p.pairs * 2 * inter * 4);
  p.out = take((size_t)p.pairs * hidden * 4);
  p.total = o;
  return true;
}
}

size_t htr_moe_scratch_bytes(int tokens, int top, int experts, int hidden, int inter) {
  MoePlan p;
  return moe_plan(tokens, top, experts, hidden, inter, p) ? p.total : 0;
}

int htr_moe_experts(const void* x, int x_dtype, const void* ids, int ids_int64, const float* weights, int tokens, int top,
                    const void* const* tensors, int experts, int hidden, int inter, int K_gate_up, int K_down, float* y,
                    void* scratch, size_t scratch_bytes, unsigned int* host_word, unsigned int ticket, void* stream) {
  if (!x || !ids || !weights || !tensors || !y) return HTR_ERR_NULL;
  if (K_gate_up < 2 || K_gate_up > 8 || K_down < 2 || K_down > 8) return HTR_ERR_K;
  if (!dtype_ok(x_dtype)) return HTR_ERR_DTYPE;
  MoePlan p;
  if (!moe_plan(tokens, top, experts, hidden, inter, p)) return HTR_ERR_SHAPE;
  if (((uintptr_t)x & 15) || ((uintptr_t)y & 15) || ((uintptr_t)ids & (ids_int64 ? 7 : 3)) || ((uintptr_t)weights & 3)) return HTR_ERR_ALIGN;
  for (int i = 0; i < experts * 8; ++i) {
    if (!tensors[i]) return HTR_ERR_NULL;
    if ((uintptr_t)tensors[i] & ((i & 3) == 0 ? 15 : ((i & 3) == 1 ? 1 : 0))) return HTR_ERR_ALIGN;
  }
  if (!scratch || scratch_bytes < p.total || ((uintptr_t)scratch & 255)) return HTR_ERR_WORKSPACE;
  unsigned char* base = (unsigned char*)scratch;
  hipStream_t st = (hipStream_t)stream;
  const void** table = (const void**)(base + p.table);
  MoePtrs ptrs;
  auto addresses = [&](int e0, int count) {
    memcpy(&ptrs, tensors + (size_t)e0 * 8, (size_t)count * 64);
    memset((unsigned char*)&ptrs + (size_t)count * 64, 0, sizeof(ptrs) - (size_t)count * 64);
  };
  const bool given = experts <= MOE_PTR_CHUNK;                    // the routing kernel takes the addresses itself
  for (int e0 = 0; !given && e0 < experts; e0 += MOE_PTR_CHUNK) {
    const int count = experts - e0 < MOE_PTR_CHUNK ? experts - e0 : MOE_PTR_CHUNK;
    addresses(e0, count);
    HTR_CHECK_HIP(launch_kernel(k_moe_experts, dim3(1), dim3(MOE_PTR_CHUNK * 8), 0, st, ptrs, table, e0, count));
  }
  addresses(0, given ? experts : 0);
  MoeRoute r;
  r.ids = ids; r.ids64 = ids_int64; r.pairs = p.pairs; r.top = top; r.experts = experts; r.entries = p.entries; r.rows_per_entry = p.rows;
  r.table = table; r.m1 = 2 * inter; r.m2 = hidden;
  r.e1 = (htr_group_entry*)(base + p.e1); r.e2 = (htr_group_entry*)(base + p.e2);
  r.h = (float*)(base + p.h); r.out = (float*)(base + p.out);
  r.pos_of = (int*)(base + p.pos); r.info = (int4*)(base + p.info);
  r.host_word = host_word; r.ticket = ticket;
  HTR_CHECK_HIP(given ? launch_kernel(k_moe_route<true>, dim3(1), dim3(MOE_ROUTE_THREADS), 0, st, r, ptrs)
                      : launch_kernel(k_moe_route<false>, dim3(1), dim3(MOE_ROUTE_THREADS), 0, st, r, ptrs));
  LinearTail t1 = {}, t2 = {};
  t1.xt_g = (const _Float16*)(base + p.xt1); t1.xs_g = (const float*)(base + p.xs1); t1.sc_g = (const float*)(base + p.sc1);
  t2.xt_g = (const _Float16*)(base + p.xt2); t2.xs_g = (const float*)(base + p.xs2); t2.sc_g = (const float*)(base + p.sc2);
  t1.cbscale = t2.cbscale = htr_cbscale();
  t1.group = r.e1; t2.group = r.e2;
  HTR_CHECK_HIP(launch_kernel(k_moe_rotate, dim3(moe_rotate_grid(p.pairs)), dim3(256), 0, st, x, x_dtype, p.pairs, (const int4*)r.info, (const void* const*)table, hidden,
                              (_Float16*)t1.xt_g, (float*)t1.xs_g, (float*)t1.sc_g));
  const int flags = HTR_F32 << 2 | FLAG_ENTRY_TILES;
  BatchArgs b1 = {nullptr, nullptr, nullptr, nullptr, 2 * inter, hidden, 0, flags}, b2 = {nullptr, nullptr, nullptr, nullptr, hidden, inter, 0, flags};
  int rc = HTR_OK;
  if (p.rows == 32) { HTR_FOR_K(K_gate_up, rc = (launch_tile_v<KK, 1, true>(b1, t1, 1, p.entries, st))); }
  else { HTR_FOR_K(K_gate_up, rc = (launch_tile_v<KK, 2, true>(b1, t1, 1, p.entries, st))); }
  if (rc != HTR_OK) return rc;
  HTR_CHECK_HIP(launch_kernel(k_moe_act, dim3(moe_rotate_grid(p.pairs)), dim3(256), 0, st, (const float*)r.h, x_dtype, p.pairs, (const int4*)r.info,
                              (const void* const*)table, inter, (_Float16*)t2.xt_g, (float*)t2.xs_g, (float*)t2.sc_g));
  if (p.rows == 32) { HTR_FOR_K(K_down, rc = (launch_tile_v<KK, 1, true>(b2, t2, 1, p.entries, st))); }
  else { HTR_FOR_K(K_down, rc = (launch_tile_v<KK, 2, true>(b2, t2, 1, p.entries, st))); }
  if (rc != HTR_OK) return rc;
  HTR_CHECK_HIP(launch_kernel(k_moe_combine, dim3(tokens, (hidden / 4 + 255) / 256), dim3(256), 0, st, (const float*)r.out, (const int*)r.pos_of,
                              weights, top, hidden, y));
  return HTR_OK;
}

// ---- timing anchors (measurement only; see the kernels).  kind 1: htr_linear's launch for one bf16 / f16 row with the
// decode compiled out; kind 2: only the weight stream of that launch.  Same plan, grid and LDS request as htr_linear.
int htr_anchor_linear(int kind, const void* qweight, const void* scales, const void* su, const void* sv, const void* x, void* y,
                      int m, int n, int K, int x_dtype, int y_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  if (!qweight || !scales || !su || !sv || !x || !y) return HTR_ERR_NULL;
  if (K != 4 || (kind != 1 && kind != 2)) return HTR_ERR_K;
  if (!shape_ok(m, n)) return HTR_ERR_SHAPE;
  if (x_dtype == HTR_F32 || !dtype_ok(x_dtype) || !dtype_ok(y_dtype)) return HTR_ERR_DTYPE;
  if (((uintptr_t)qweight & 15) || ((uintptr_t)x & 3)) return HTR_ERR_ALIGN;
  Plan pl;
  if (!make_plan(m, n, K, 1, 0, pl) || pl.prerot) return HTR_ERR_SPLIT;
  const size_t need = htr_workspace_bytes(m, n, K, 1, 0);
  if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 255)) return HTR_ERR_WORKSPACE;
  LinearLaunch a;
  a.qw = (const uint32_t*)qweight; a.x = x; a.su = (const uint8_t*)su;
  a.part = (float*)((unsigned char*)workspace + WS_HEADER);
  a.m = m; a.n = n; a.M = 1; a.chunk = pl.chunk; a.flags = x_dtype | (y_dtype << 2); a.problems = 1;
  const int nblk = n / 128, rbs = m / 128;
  if (pl.chunk < nblk && nblk % pl.chunk == 0 && rbs % 8 == 0 && rbs >= 16 && pl.wgs % 8 == 0) a.flags |= FLAG_LANES | ((pl.wgs / 8) << FLAG_LANE_LEN_SHIFT);
  a.nblk_magic = (((unsigned long long)1 << 40) + (unsigned)nblk - 1) / (unsigned)nblk;
  LinearTail& t = a.tail;
  t.scales = (const uint16_t*)scales; t.sv = (const uint8_t*)sv; t.bias = nullptr; t.y = y;
  t.xt_g = nullptr; t.xs_g = nullptr; t.sc_g = nullptr;
  t.status = (uint32_t*)workspace;
  t.cbscale = htr_cbscale();
  t.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
  t.group = nullptr; t.group_prerot_stride = 0; t.group_part_stride = 0; t.tiles = nullptr;
  t.chunk_magic = (((unsigned long long)1 << 40) + (unsigned)pl.chunk - 1) / (unsigned)pl.chunk;
  hipStream_t st = (hipStream_t)stream;
  const size_t lds = balanced_lds_request(pl.lds, pl.wgs);
  if (kind == 2) {
    HTR_CHECK_HIP(launch_kernel(k_anchor_read<4, 4>, dim3(pl.wgs), dim3(WG_THREADS), lds, st, a.qw, m, n, a.chunk, a.flags, a.nblk_magic,
                                (uint32_t*)((unsigned char*)workspace + ws_half(workspace_bytes))));
    return HTR_OK;
  }
  if (pl.chunk <= 8) {
    HTR_CHECK_HIP((allow_full_lds<k_linear<4, 1, 4, 4, false, 1, 1>>()));
    HTR_CHECK_HIP(launch_kernel(k_linear<4, 1, 4, 4, false, 1, 1>, dim3(pl.wgs), dim3(WG_THREADS), lds, st, a.qw, a.x, a.su, a.part,
                                a.m, a.n, a.M, a.chunk, a.flags, a.nblk_magic, a.tail));
  } else {
    HTR_CHECK_HIP((allow_full_lds<k_linear<4, 1, 4, 2, false, 1, 1>>()));
    HTR_CHECK_HIP(launch_kernel(k_linear<4, 1, 4, 2, false, 1, 1>, dim3(pl.wgs), dim3(WG_THREADS), lds, st, a.qw, a.x, a.su, a.part,
                                a.m, a.n, a.M, a.chunk, a.flags, a.nblk_magic, a.tail));
  }
  return HTR_OK;
}

// The decode of one wave-step (2048 weights) on register data: `workgroups` workgroups of 8 waves, one per compute unit
// (two waves per SIMD, as in the batch-1 launches), `iters` wave-steps each; out_u64[2 * wave] = shader-clock cycles,
// out_u64[2 * wave + 1] = ticks of the 100 MHz reference clock over the loop.
int htr_anchor_decode(int K, int with_mfma, int iters, int workgroups, void* out_u64, void* stream) {
  if (!out_u64) return HTR_ERR_NULL;
  if (K < 2 || K > 5) return HTR_ERR_K;
  if (iters < 1 || workgroups < 1 || workgroups > 65536) return HTR_ERR_SHAPE;
  hipStream_t st = (hipStream_t)stream;
  const size_t lds = balanced_lds_request(1024, workgroups <= num_cu() ? num_cu() : workgroups);
#define HTR_LAUNCH_ANCHOR(KK_, MF_)                                                                                          \
  {                                                                                                                          \
    HTR_CHECK_HIP((allow_full_lds<k_anchor_decode<KK_, MF_>>()));                                                            \
    HTR_CHECK_HIP(launch_kernel(k_anchor_decode<KK_, MF_>, dim3(workgroups), dim3(WG_THREADS), lds, st, iters,               \
                                (unsigned long long*)out_u64, (float*)nullptr));                                             \
  }
  switch (K) {
    case 2: if (with_mfma) HTR_LAUNCH_ANCHOR(2, true) else HTR_LAUNCH_ANCHOR(2, false) break;
    case 3: if (with_mfma) HTR_LAUNCH_ANCHOR(3, true) else HTR_LAUNCH_ANCHOR(3, false) break;
    case 4: if (with_mfma) HTR_LAUNCH_ANCHOR(4, true) else HTR_LAUNCH_ANCHOR(4, false) break;
    default: if (with_mfma) HTR_LAUNCH_ANCHOR(5, true) else HTR_LAUNCH_ANCHOR(5, false) break;
  }
#undef HTR_LAUNCH_ANCHOR
  return HTR_OK;
}

// workgroups of a search: one per compute unit at most, each takes tiles in turn and keeps its stored arrays in a slot of its own
static unsigned viterbi_grid(int64_t tiles) { const int cus = num_cu(); return (unsigned)(tiles < cus ? tiles : cus); }

size_t htr_viterbi_workspace_bytes(int64_t tiles, int T, int K) {
  if (tiles <= 0 || T < 1 || T > 256 || K < 2 || K > 8) return 0;
  size_t rows = 0;
  HTR_FOR_K_OR(K, rows = (size_t)vit_rows(T, VitCfg<KK>::C), return 0);
  return align256(viterbi_grid(tiles) * (rows > 0 ? rows : 1) * (65536u >> K) * sizeof(float)) + 16;      // 16: any start will do
}

int htr_viterbi(const void* x, const void* w, int64_t tiles, int T, int K, int tailbite, void* states_u16, void* workspace,
                size_t workspace_bytes, void* stream) {
  if (!x || !w || !states_u16) return HTR_ERR_NULL;
  if (K < 2 || K > 8) return HTR_ERR_K;
  if (tiles <= 0 || tiles > 0x7FFFFFFF || T < 1 || T > 256) return HTR_ERR_SHAPE;
  if (((uintptr_t)x & 3) || ((uintptr_t)w & 3) || ((uintptr_t)states_u16 & 1)) return HTR_ERR_ALIGN;
  const size_t need = htr_viterbi_workspace_bytes(tiles, T, K);
  if (!workspace || workspace_bytes < need) return HTR_ERR_WORKSPACE;
  workspace = (void*)(((uintptr_t)workspace + 15) & ~(uintptr_t)15);
  hipStream_t st = (hipStream_t)stream;
  const double rms = __builtin_sqrt(MEAN_SQ);
#define HTR_LAUNCH_VIT(KK_)                                                                                              \
  {                                                                                                                      \
    HTR_CHECK_HIP((allow_full_lds<k_viterbi<KK_>>()));                                                                   \
    HTR_CHECK_HIP(launch_kernel(k_viterbi<KK_>, dim3(viterbi_grid(tiles)), dim3(VitCfg<KK_>::THREADS), VitCfg<KK_>::LDS, st, \
                                (const float*)x, (const float*)w, (int)tiles, T, tailbite ? 1 : 0, (float*)workspace,    \
                                (uint16_t*)states_u16, rms));                                                            \
  }
  HTR_FOR_K(K, HTR_LAUNCH_VIT(KK));
#undef HTR_LAUNCH_VIT
  return HTR_OK;
}

static int encode_block_args(const void* const* pointers, int count, int64_t rows, int64_t n, int64_t col) {
  for (int i = 0; i < count; ++i) {
    if (!pointers[i]) return HTR_ERR_NULL;
    if ((uintptr_t)pointers[i] & 15) return HTR_ERR_ALIGN;
  }
  if (rows <= 0 || rows % 16 || rows > ((int64_t)1 << 30) || n <= 0 || n % 16 || n > ((int64_t)1 << 30) || col < 0 || col % 16 || col >= n) return HTR_ERR_SHAPE;
  return HTR_OK;
}

int htr_encode_targets(const void* W, const void* F, const void* scales, int64_t rows, int64_t n, int64_t col, void* x, void* stream) {
  const void* pointers[] = {W, F, scales, x};
  const int rc = encode_block_args(pointers, 4, rows, n, col);
  if (rc != HTR_OK) return rc;
  HTR_CHECK_HIP(launch_kernel(k_encode_targets, dim3((unsigned)((rows * 4 + 255) / 256)), dim3(256), 0, (hipStream_t)stream, (const float*)W,
                              (const float*)F, (const float*)scales, rows, n, col, (float*)x));
  return HTR_OK;
}

int htr_encode_quantized(const void* states_u16, const void* codebook, const void* W, const void* scales, int64_t rows, int64_t n, int64_t col,
                         void* Q, void* err, void* states_i64, void* stream) {
  const void* pointers[] = {states_u16, codebook, W, scales, Q, err, states_i64};
  const int rc = encode_block_args(pointers, 7, rows, n, col);
  if (rc != HTR_OK) return rc;
  HTR_CHECK_HIP(launch_kernel(k_encode_quantized, dim3((unsigned)((rows * 4 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                              (const uint16_t*)states_u16, (const float*)codebook, (const float*)W, (const float*)scales, rows, n, col, (float*)Q,
                              (float*)err, (int64_t*)states_i64));
  return HTR_OK;
}

int htr_decode_raw(const void* qweight, void* out_i16, int64_t ntiles, int K, void* stream) {
  if (!qweight || !out_i16) return HTR_ERR_NULL;
  if (K < 2 || K > 8) return HTR_ERR_K;
  if (ntiles <= 0) return HTR_ERR_SHAPE;
  if (((uintptr_t)qweight & 15) || ((uintptr_t)out_i16 & 15)) return HTR_ERR_ALIGN;
  const int64_t blocks = (ntiles * 8 + 255) / 256;
  hipStream_t st = (hipStream_t)stream;
  HTR_FOR_K(K, HTR_CHECK_HIP(launch_kernel(k_decode_raw<KK>, dim3((unsigned)blocks), dim3(256), 0, st, (const uint32_t*)qweight,
                                           (int16_t*)out_i16, ntiles)));
  return HTR_OK;
}

int htr_dequant_w(const void* qweight, const void* scales, const void* su, const void* sv, void* out_bf16, int m, int n,
                  int K, void* stream) {
  if (!qweight || !scales || !su || !sv || !out_bf16) return HTR_ERR_NULL;
  if (K < 2 || K > 8) return HTR_ERR_K;
  if (m <= 0 || n <= 0 || m % 128 || n % 128 || m / 128 > 65535) return HTR_ERR_SHAPE;
  if (((uintptr_t)qweight & 15) || ((uintptr_t)out_bf16 & 3) || ((uintptr_t)scales & 1) || ((uintptr_t)sv & 3)) return HTR_ERR_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid(n / 128, m / 128);
  const size_t lds = DQW_LDS;
  const float cb = htr_cbscale();
#define HTR_LAUNCH_DQW(KK_)                                                                                              \
  {                                                                                                                      \
    HTR_CHECK_HIP((allow_full_lds<k_dequant_w<KK_>>()));                                                                 \
    HTR_CHECK_HIP(launch_kernel(k_dequant_w<KK_>, grid, dim3(512), lds, st, (const uint32_t*)qweight, (const uint16_t*)scales, \
                                (const uint8_t*)su, (const uint8_t*)sv, (uint16_t*)out_bf16, n / 16, cb));               \
  }
  HTR_FOR_K(K, HTR_LAUNCH_DQW(KK));
#undef HTR_LAUNCH_DQW
  return HTR_OK;
}

int htr_dequant_q(const void* qweight, const void* scales, void* out_f32, int mt, int nt, int K, void* stream) {
  if (!qweight || !scales || !out_f32) return HTR_ERR_NULL;
  if (K < 2 || K > 8) return HTR_ERR_K;
  if (mt <= 0 || nt <= 0) return HTR_ERR_SHAPE;
  if (((uintptr_t)qweight & 15) || ((uintptr_t)out_f32 & 3) || ((uintptr_t)scales & 1)) return HTR_ERR_ALIGN;
  const int64_t blocks = ((int64_t)mt * nt * 8 + 255) / 256;
  hipStream_t st = (hipStream_t)stream;
  const double rms = __builtin_sqrt(MEAN_SQ);
  HTR_FOR_K(K, HTR_CHECK_HIP(launch_kernel(k_dequant_q<KK>, dim3((unsigned)blocks), dim3(256), 0, st, (const uint32_t*)qweight,
                                           (const uint16_t*)scales, (float*)out_f32, mt, nt, rms)));
  return HTR_OK;
}

}  // extern "C"
