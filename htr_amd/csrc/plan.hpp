// Part of htr_gfx950.hip, included inside its anonymous namespace: workspace layout, launch plans and launchers (host side).
// ------------------------------------------------------------------------------------------------ workspace set-up
// Zeroes the first `bytes` (a multiple of 16) of a workspace and writes the header's mirror address.  A kernel, not a
// memset, so that it can be recorded into a HIP graph.
__global__ __launch_bounds__(256) void k_workspace_init(u4* __restrict__ ws, size_t bytes, unsigned long long mirror) {
  const size_t n16 = bytes / 16;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += (size_t)gridDim.x * 256)
    ws[i] = i == 0 ? u4{0u, 0u, (uint32_t)mirror, (uint32_t)(mirror >> 32)} : u4{0u, 0u, 0u, 0u};
}

// ------------------------------------------------------------------------------------------------ host side
thread_local int g_last_hip_error = 0;
std::atomic<int> g_spin_limit{1 << 20};     // polls (about a microsecond each) before a finishing workgroup gives up

struct Plan { int chunk, wgs, segfin, nbl, mb, prerot; size_t lds; };

// Workspace: two halves, split at workspace_bytes / 2 (rounded down to 256).  First half: [256-byte header: status
// word][one partial slot per workgroup]; it must be all-zero between calls.  Second half: scratch for the pre-rotated
// activations, left as it is.  The split depends only on the size the caller passes, not on the problem, so no call can
// leave scratch data where a later call of another shape expects zeroed slots (as long as the caller passes the same
// size with the same buffer).
constexpr size_t WS_HEADER = 256;
inline size_t align256(size_t v) { return (v + 255) / 256 * 256; }
inline size_t ws_need(size_t slot_bytes, size_t scratch_bytes) {
  const size_t a = align256(WS_HEADER + slot_bytes), b = align256(scratch_bytes);
  return 2 * (a > b ? a : b);
}
inline size_t ws_half(size_t workspace_bytes) { return workspace_bytes / 2 / 256 * 256; }
// bytes of the pre-rotated activations, their block sums and the row scales
inline size_t prerot_bytes(int n, size_t M) { return align256(M * n * 2) + align256(M * (n / 128) * 16) + align256(M * 4); }
inline void place_prerot(LinearTail& t, unsigned char* at, int n, size_t M) {
  t.xt_g = (const _Float16*)at;
  t.xs_g = (const float*)(at + align256(M * n * 2));
  t.sc_g = (const float*)(at + align256(M * n * 2) + align256(M * (n / 128) * 16));
}

// ---- facts of the device the plans are made for: compute units and LDS bytes per compute unit, read once per device
// (the current one) from the runtime; an unpartitioned MI355X (256 CUs, 160 KB) where no device can be asked (plans
// computed on a machine without a GPU).  htr_plan_device_override replaces them for every device (tests, tuning).
struct DeviceFacts { int cus; size_t lds; };
constexpr int MAX_DEVICES = 64;
constexpr DeviceFacts MI355X_FACTS = {256, 160 * 1024};
std::atomic<int> g_override_cus{0};
std::atomic<long> g_override_lds{0};
inline DeviceFacts device_facts() {
  static DeviceFacts table[MAX_DEVICES];
  static std::atomic<uint64_t> known{0};
  const int ov = g_override_cus.load(std::memory_order_acquire);
  if (ov > 0) return DeviceFacts{ov, (size_t)g_override_lds.load(std::memory_order_acquire)};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) { (void)hipGetLastError(); return MI355X_FACTS; }
  if (dev < 0 || dev >= MAX_DEVICES) return MI355X_FACTS;
  const uint64_t bit = (uint64_t)1 << dev;
  if (known.load(std::memory_order_acquire) & bit) return table[dev];
  int cus = 0, lds = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1 ||
      hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) != hipSuccess || lds < 64 * 1024) {
    (void)hipGetLastError();
    return MI355X_FACTS;
  }
  table[dev] = DeviceFacts{cus, (size_t)lds};        // two threads racing here store the same values
  known.fetch_or(bit, std::memory_order_release);
  return table[dev];
}
inline int num_cu() { return device_facts().cus; }
constexpr int MAX_ROW_BLOCKS = 16384;
constexpr int MAX_CHUNK = 4096;
// the kernel divides step indices by n / 128 with a 40-bit reciprocal: exact while indices stay below 2^24
inline bool shape_ok(int m, int n) {
  return m > 0 && n > 0 && m % 128 == 0 && n % 128 == 0 && m / 128 <= MAX_ROW_BLOCKS && n / 128 < 65536 &&
         (long)(m / 128) * (n / 128) < (1L << 24) - 2 * MAX_CHUNK;
}

inline bool plan_for_chunk(int m, int n, int M, int chunk, Plan& pl) {
  const int nblk = n / 128, rbs = m / 128;
  const long vtotal = (long)rbs * nblk;
  if (chunk < 1 || chunk > vtotal || chunk > MAX_CHUNK) return false;
  pl.chunk = chunk;
  pl.wgs = (int)((vtotal + chunk - 1) / chunk);
  pl.segfin = (chunk + nblk - 1) / nblk;            // row blocks that can end inside one chunk
  pl.nbl = chunk < nblk ? chunk : nblk;
  pl.lds = lds_bytes(M, pl.nbl, pl.segfin);
  if (pl.lds > (size_t)LDS_BUDGET) return false;
  // a workgroup rotates its own column blocks while that is at most ROT_PAIRS (row, block) pairs (MAX_ROT_PAIRS with up
  // to eight rows: the kernel variant with several passes); beyond that the activations are rotated once, ahead of
  // the launch
  pl.prerot = M * pl.nbl > (M <= 8 ? MAX_ROT_PAIRS : ROT_PAIRS) ? 1 : 0;
  return true;
}

// Picks the chunk length (virtual steps per workgroup) with a cost model in microseconds fitted to chunk-length sweeps
// on MI355X (K4, 1..8 rows, nine shapes from 1024x4096 to 28672x4096, twenty chunk lengths each; the choice is within
// 1 % of the best measured chunk on average, 10 % at worst): a fixed latency chain (launch, x fetch, rotation, partial
// exchange, output rotation) that grows with the contributors a finisher reads, eight per round trip; a cost per
// step that depends on how many workgroups share a CU (one: the workgroup's own decode rate, 0.4 .. 0.5 us; several:
// throughput bound, proportional to the load of the fullest CU, plus a set-up per workgroup); a penalty for chunks
// that do not tile the rows of column blocks; the extra launch of a pre-rotation; and the growth of all per-step work
// with the number of activation rows.
inline bool search_chunk(int m, int n, int M, int cus, Plan& pl) {
  const int nblk = n / 128, rbs = m / 128;
  const long vtotal = (long)rbs * nblk;
  const double rows = M <= 8 ? 1.0 + 0.06 * (M - 1) : (M <= 16 ? 2.2 : 6.5);
  double best = 1e30;
  bool found = false;
  const int max_chunk = (int)(vtotal < MAX_CHUNK ? vtotal : MAX_CHUNK);
  for (int chunk = 1; chunk <= max_chunk; ++chunk) {
    Plan c;
    c.mb = pl.mb;
    if (!plan_for_chunk(m, n, M, chunk, c)) continue;
    const double fill = (double)c.wgs / cus;
    const bool aligned = (nblk % chunk == 0) || (chunk % nblk == 0);
    const int contributors = chunk >= nblk ? 1 : (nblk + chunk - 1) / chunk;
    const double steps = chunk * (aligned ? 1.0 : 1.06 + 0.04 * (M - 1));
    // one workgroup per CU or fewer: the chip works through `chunk` steps once; more: the fullest CU works through
    // its workgroups one after the other, each with its own set-up and partial hand-over
    // (a grid slightly above one workgroup per CU leaves a few CUs with two: it costs nearly as much as two everywhere)
    const double fill2 = fill < 1.5 ? 1.5 : fill;
    const double body = fill <= 1.0 ? rows * (0.4 + 0.05 * fill) * steps
                                    : fill2 * (rows * 0.55 * steps + 0.5 + 0.1 * M);
    // hand-over: the contributors' slots are read eight per round trip to memory (0.45 us each)
    const double handover = 0.45 * ((contributors - 1 + 7) / 8);
    const int passes = (M * c.nbl + ROT_PAIRS - 1) / ROT_PAIRS;      // rotation passes inside the kernel, 0.3 us each after the first
    const double t = 4.5 + handover + (c.prerot ? 3.0 + 0.1 * M : 0.3 * (passes - 1)) + body;
    if (t < best) { best = t; pl = c; found = true; }
  }
  return found;
}

inline bool search_plan(int m, int n, int K, int M, int nsplit, int cus, Plan& pl) {
  const int nblk = n / 128, rbs = m / 128;
  const long vtotal = (long)rbs * nblk;
  pl.mb = M <= 8 ? 1 : (M <= 16 ? 2 : 4);
  if (nsplit > 0) {                                                 // explicit plan (tuning): chunk length in the low
    const int chunk = nsplit & 0xFFFFF;                             // 20 bits, bit 30 = force pre-rotation
    bool ok = chunk > 0 ? plan_for_chunk(m, n, M, chunk, pl) : false;
    if (ok && (nsplit & (1 << 30))) pl.prerot = 1;
    return ok;
  }
  // Large matrices: one row block per workgroup where that fits LDS
  const bool large = vtotal >= (long)64 * cus && nblk <= 64;
  bool found = false;
  if (large) {
    Plan whole;
    whole.mb = pl.mb;
    found = plan_for_chunk(m, n, M, nblk, whole);
    if (found) pl = whole;
  }
  if (!found) found = search_chunk(m, n, M, cus, pl);
  // ... or, instead of either, two equal chunks per compute unit.  The compute units take workgroups in rounds, so the last round is as
  // long as the others however few are left; equal chunks fill it, at the price of partials, of row ends inside a chunk, and of PACE
  // where the activations are rotated ahead.  They pay where the rounds hold `spare` times the steps that there are: later from five
  // bits on, as whole row blocks then read at close to the memory's rate already (61184x6144 K5 4.4, K8 4.9 of the 5.0 TB/s of a copy;
  // K4 3.7), though up to K6 not over short rows, nor with more rounds, whose workgroups each pay for their ends.  Measured on MI355X
  // with margins from 1.005 to 1.5, n from 1536 to 8192, two to eleven rounds; us with row blocks / chunks at a margin:
  //   K4 1 row 63616x6144 (1.03) 48.8 / 50.8, 61824x6144 (1.06) 50.6 / 50.6, 60032x6144 (1.09) 49.0 / 47.0; five rounds 158976x4096
  //   (1.03) 77.0 / 75.4, 152064x4096 (1.08) 72.8 / 71.7; three 73728x4096 (1.33) 48.6 / 39.8; 5 rows, rotated ahead, 92672x4096 (1.06)
  //   52.9 / 53.4, 90112x4096 (1.09) 52.5 / 50.9
  //   K5 1 row 122496x2560 (1.07) 45.8 / 45.0, K6 153088x2048 (1.07) 54.1 / 51.6: short rows
  //   K5 1 row 61184x6144 (1.07) 53.2 / 53.8, 3 rows, rotated ahead, 60032x6144 (1.09) 55.1 / 58.3, 5 rows 84736x4096 (1.16) 57.1 / 58.9
  //   K6 1 row 61184x5120 (1.07) 51.1 / 52.8, 3 rows 112896x3072 (1.16) 60.4 / 56.5; K7 1 row 93568x4096 (1.05) 66.7 / 69.6; K8 3 rows
  //   87680x3072 (1.12) 58.1 / 59.2
  //   five rounds, 1 row 151680x4096 (1.08) K5 83.3 / 81.4, K6 94.3 / 91.9, K7 104.2 / 106.5; K8 5 rows 116992x3072 (1.12) 75.4 / 79.1; K5 5
  //   rows, rotated ahead, 151680x4096 89.3 / 91.5, 147584x4096 89.2 / 89.9
  //   3 rows of 8192, whose row blocks do not fit, with the search's 32 steps: K4 61184 (1.07) 66.6 / 64.6, 43648 (1.12) 51.4 / 49.1; K6
  //   46720 (1.05) 63.7 / 67.1, 50304 (1.30) 79.1 / 74.3; K7 46720 72.1 / 77.2
  Plan even;
  even.mb = pl.mb;
  if (large && plan_for_chunk(m, n, M, (int)((vtotal + 2 * cus - 1) / (2 * cus)), even)) {
    const int rounds = (rbs + cus - 1) / cus;
    double spare;
    if (K <= 4) spare = rounds >= 3 ? 1.03 : 1.06;
    else if (K <= 6 && K * nblk <= 120) spare = 1.03;
    else spare = K <= 6 && rounds >= 4 ? 1.06 : 1.15;
    if (even.prerot && (K > 4 || pl.chunk == nblk)) spare += 0.07;
    // partials beyond the library's own workspace (4 rows of 262144 and more), which two slots per compute unit always fit: 437888x3584
    // K6 4 rows 278.8 / 251.9, 310272x4096 K4 171.9 / 161.4
    const double fitting = even.prerot && M > 4 ? 1.1 : 1.03;
    if (found && spare > fitting && ws_need((size_t)pl.wgs * M * 128 * sizeof(float), prerot_bytes(n, M)) > HTR_STATIC_SCRATCH_BYTES) spare = fitting;
    if (!found || spare * vtotal < (double)((pl.wgs + cus - 1) / cus) * pl.chunk * cus) { pl = even; found = true; }
  }
  return found;
}

// The search above walks every chunk length (up to 4096 of them): tens of microseconds on the host, more than the launch
// it plans.  Plans depend only on (m, n, K, M, nsplit) and the device's CU count, so the last 64 distinct ones are kept.
inline bool make_plan(int m, int n, int K, int M, int nsplit, Plan& pl) {
  const int cus = num_cu();
  struct Entry { int m, n, K, M, nsplit, cus; bool ok; Plan pl; };
  static Entry cache[64];
  static int filled = 0, next = 0;
  static std::atomic_flag busy = ATOMIC_FLAG_INIT;
  while (busy.test_and_set(std::memory_order_acquire)) {}
  for (int i = 0; i < filled; ++i) {
    const Entry& e = cache[i];
    if (e.m == m && e.n == n && e.K == K && e.M == M && e.nsplit == nsplit && e.cus == cus) {
      const bool ok = e.ok;
      pl = e.pl;
      busy.clear(std::memory_order_release);
      return ok;
    }
  }
  busy.clear(std::memory_order_release);
  Plan found = {};
  const bool ok = search_plan(m, n, K, M, nsplit, cus, found);
  while (busy.test_and_set(std::memory_order_acquire)) {}
  Entry& e = cache[next];
  e.m = m; e.n = n; e.K = K; e.M = M; e.nsplit = nsplit; e.cus = cus; e.ok = ok; e.pl = found;
  next = (next + 1) % 64;
  if (filled < 64) ++filled;
  busy.clear(std::memory_order_release);
  pl = found;
  return ok;
}

// The dispatcher places workgroups wherever resources allow, not evenly: with 512 equal workgroups some CUs receive
// three and others one, and the kernel ends with the most loaded CU.  Requesting 1/k of a CU's LDS (160 KB on MI355X) per
// workgroup (k = workgroups per CU when spread evenly) makes exactly k fit, so the spread is even.
inline size_t balanced_lds_request(size_t needed, int grid) {
  const DeviceFacts df = device_facts();
  const int k = (grid + df.cus - 1) / df.cus;
  if (k > 4) return needed;
  const size_t share = (df.lds / k) / 1024 * 1024 - 1024;
  return share > needed ? share : needed;
}

// One launch with the runtime's own return value (hipGetLastError after a launch macro would also report an earlier,
// unrelated failure of the thread as this launch's).
template <typename T> struct same_type { typedef T type; };
template <typename... KArgs>
hipError_t launch_kernel(void (*kern)(KArgs...), dim3 grid, dim3 block, size_t lds, hipStream_t st, typename same_type<KArgs>::type... args) {
  void* argv[] = {(void*)&args...};
  return hipLaunchKernel((const void*)kern, grid, block, argv, lds, st);
}
// Kernels that may ask for more than the default 48 KB of dynamic LDS get the limit raised to the whole 160 KB once per
// (kernel, device), not per launch with the launch's own value: the attribute is state of the function, and two host
// threads that set different values around their launches would race.
constexpr int MAX_DYNAMIC_LDS = 160 * 1024;
template <auto Kern> hipError_t allow_full_lds() {
  static std::atomic<uint64_t> done{0};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = (uint64_t)1 << (dev & 63);
  if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
  e = hipFuncSetAttribute((const void*)Kern, hipFuncAttributeMaxDynamicSharedMemorySize, MAX_DYNAMIC_LDS);
  if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
  return e;
}
#define HTR_CHECK_HIP(EXPR) do { hipError_t e_ = (EXPR); if (e_ != hipSuccess) { g_last_hip_error = (int)e_; return HTR_ERR_LAUNCH; } } while (0)

struct LinearLaunch {
  const uint32_t* qw; const void* x; const uint8_t* su; float* part;
  int m, n, M, chunk, flags, problems;
  unsigned long long nblk_magic;
  LinearTail tail;
};

template <int K, int MB, bool DEEP, bool PREROT, int RP = 1, bool PACE = false>
int launch_linear_v(const LinearLaunch& a, int grid, size_t lds, hipStream_t st) {
  constexpr int P = K <= 4 ? 4 : (K <= 6 ? 3 : 2);          // wave-steps of weights in flight
  constexpr int D = DEEP && P >= 4 ? 4 : 2;                 // steps decoded ahead of the activation exchange
  lds = balanced_lds_request(lds, grid * a.problems);
  HTR_CHECK_HIP((allow_full_lds<k_linear<K, MB, P, D, PREROT, RP, 0, PACE>>()));
  HTR_CHECK_HIP(launch_kernel(k_linear<K, MB, P, D, PREROT, RP, 0, PACE>, dim3(grid, a.problems), dim3(WG_THREADS), lds, st, a.qw, a.x, a.su,
                              a.part, a.m, a.n, a.M, a.chunk, a.flags, a.nblk_magic, a.tail));
  return HTR_OK;
}
// Where the two waves of a SIMD are kept in step by alternating priorities (k_linear's PACE): chunks of twelve steps and
// more, one launch (not a group), and either up to four activation rows or at most two chunks per row block.
// Measured on MI355X, K4, us without -> with: 28672x4096 1 row 19.1 -> 17.7, 4 rows 22.0 -> 20.5, 8 rows 23.3 -> 23.5;
// 14336x4096 1 / 4 / 8 rows 12.3 -> 11.8, 13.7 -> 12.9, 15.8 -> 14.4; 4096x14336 (eight chunks per row block) 1 / 4 / 6 /
// 8 rows 11.9 -> 11.2, 12.9 -> 12.7, 14.0 -> 14.1, 14.9 -> 16.0; 6144x4096 8 rows (chunks of 8) 10.0 -> 13.8.
inline bool paced(const LinearLaunch& a) {
  static const bool on = getenv("HTR_PACE") == nullptr || atoi(getenv("HTR_PACE")) != 0;
  const int nblk = a.n / 128;
  return on && a.problems == 1 && a.chunk >= 12 && (a.M <= 4 || (nblk + a.chunk - 1) / a.chunk <= 2);
}
// Short chunks are decoded completely ahead of the activation exchange (more registers, so only for one activation
// block and chunks whose prologue latency is a large part of the kernel); long chunks prefer occupancy.
template <int K, bool PREROT> int launch_linear_kr(const LinearLaunch& a, int mb, int grid, size_t lds, hipStream_t st) {
  const bool deep = a.chunk <= 8;
  if constexpr (!PREROT) {                 // more pairs than one pass rotates: the variant with several passes (up to 8 rows)
    const int nblk = a.n / 128;
    if (mb == 1 && a.M * (a.chunk < nblk ? a.chunk : nblk) > ROT_PAIRS)
      return paced(a) ? launch_linear_v<K, 1, false, false, MAX_ROT_PASSES, true>(a, grid, lds, st)
                      : launch_linear_v<K, 1, false, false, MAX_ROT_PASSES>(a, grid, lds, st);
    if (mb == 1 && !deep && paced(a)) return launch_linear_v<K, 1, false, false, 1, true>(a, grid, lds, st);
  }
  switch (mb) {
    case 1: return deep ? launch_linear_v<K, 1, true, PREROT>(a, grid, lds, st) : launch_linear_v<K, 1, false, PREROT>(a, grid, lds, st);
    case 2: return launch_linear_v<K, 2, false, PREROT>(a, grid, lds, st);
    default: return launch_linear_v<K, 4, false, PREROT>(a, grid, lds, st);
  }
}
template <int K> int launch_linear_k(const LinearLaunch& a, bool prerot, int mb, int grid, size_t lds, hipStream_t st) {
  return prerot ? launch_linear_kr<K, true>(a, mb, grid, lds, st) : launch_linear_kr<K, false>(a, mb, grid, lds, st);
}

// ---- batched kernel: split S of the column blocks per row block
struct BatchPlan { int S, cb, wgs, mb, rot, last_finishes; bool tile; size_t lds; };      // tile: k_linear_tile, unless rot
// rows x column blocks per split up to which a workgroup of the batched kernel always rotates its own activations (its ROT = 1: up to
// two units of 16 rows and one block per wave) instead of a rotation launch: 16 x 16 or 32 x 8
inline bool batch_rot_fits(int M, int cb) { return (M <= 16 && cb <= 16) || (M <= 32 && cb <= 8); }
// Where it does so beyond that with up to four units per wave (ROT = 2).  Decided at the launch, by the activations it is given; the
// plan is that of the rotation launch and of the kernel behind it, which all other activations take.  The units are of 16 rows, so
// what the workgroups spend does not grow from 17 to 32 rows, while what the launch and the kernel behind it take does not pay for
// rows that are not there: the more rows, the fewer column blocks.  More bits hide more of it, and on the smallest grids, up to a few
// row blocks, the launch is short.  Measured on MI355X, us in graphs over several weights, rotation launch / 2:
//   up to 16 rows, everywhere (28672x4096, 16 rows K4 23.9 / 23.7, 9 rows K3 23.2 / 22.1; 4096x22528, 12 rows K4 22.0 / 18.9; 128x16384,
//     16 rows K5 15.9 / 15.2)
//   17 to 32 rows over 9 and 10 column blocks, everywhere (28672x1152, 32 rows K4 14.5 / 13.9; 10240x3840 16.2 / 15.4), and from seven
//     bits on over up to 16 (128x16384, 32 rows K7 21.0 / 20.3; 20480x2048 K8 22.4 / 22.6)
//   K5 and K6: up to 20 rows (20480x2048, 17 rows K5 18.9 / 18.7, 24 and 32 rows 18.9 / 19.3 and 19.6 / 20.2); beyond, on an eighth of
//     the chip and more (128x11264, 32 rows K5 15.8 / 16.0), with four column splits and more (8192x8192, 24 rows 23.5 / 23.2, 32 rows
//     24.4 / 24.1), else over up to 14 blocks to 24 rows and then with two splits over up to 12 (28672x1664, one split over 13, 24 rows
//     17.5 / 17.4, 32 rows 18.2 / 18.4)
//   up to K4: 20 rows over 11 and 12 (14336x3072, 17 / 24 / 32 rows K4 16.7 / 16.5, 17.0 / 17.0, 16.9 / 17.3; 20480x1408, 32 rows 14.8 /
//     15.4), and 13 and 14 on a grid of three splits and more that fills three quarters of the chip (4096x14336, 24 rows K4 19.8 /
//     19.3, K3 19.1 / 18.9; K2, whose decode hides least, 17.4 / 17.4 with 17, 18.3 / 18.7 with 32)
inline bool batch_rot_long(int K, int M, int S, int cb, int wgs) {
  const int cus = num_cu();
  if (M > 32 || wgs > cus || (M <= 16 ? cb : 2 * cb) > 32) return false;
  if (M <= 16 || cb <= 10 || K >= 7) return true;
  const bool eighth = 8 * wgs >= cus;
  if (K >= 5) return M <= 20 || (eighth && (S >= 4 || (M <= 24 ? cb <= 14 : S > 1 && cb <= 12)));
  if (cb <= 12) return M <= 20 && eighth;
  return cb <= 14 && S >= 3 && 4 * wgs > 3 * cus && (K >= 3 || M <= 20);
}
constexpr int BATCH_MIN_M = 9;      // rows from which the library policy takes the batched kernel on every shape
inline int batch_groups(int M) { return M <= 16 ? 1 : (M <= 32 ? 2 : (M <= 64 ? 4 : 8)); }   // groups of 16 activation rows
// k_linear_tile instead of k_linear_batch for 17 to 64 activation rows that were rotated ahead.  Measured on MI355X, us of the call
// with its rotation, k_linear_batch / k_linear_tile:
//   more row blocks than compute units, one split: 33..64 rows, two workgroups per compute unit, always (65536x4096, 33 rows K4
//     66.8 / 50.5, K5 64.0 / 61.8, K8 76.8 / 74.0; 40960x1024, 64 rows K4 29.5 / 22.0); 17..32 rows up to K4 (65536x4096, 32 rows
//     47.8 / 45.5) and, at more bits, whose decode the two workgroups cannot hide behind each other, up to 16 column blocks
//     (65536x4096, 32 rows K5 52.2 / 56.9, 40960x2048 K5 29.8 / 29.8, 65536x1024 K5 22.5 / 20.5)
//   else up to K4 from 14 column blocks per split (28672x4096, 33 rows K4 33.6 / 30.5; 14336x4096 21.8 / 20.9; 10240x4096 with 11
//     blocks, 48 rows 19.5 / 20.1, 4096x4096 with 4, 33 rows 12.5 / 13.2; 28672x4096, 64 rows K5 36.5 / 41.5)
//   and up to two splits: with more, single calls are ahead (4096x14336, eight splits, 33 rows K3 22.1 / 20.8), but whole layers
//     are not, where the launch follows a larger one.  Graphs of six layers, us, k_linear_batch throughout / k_linear_tile for any
//     number of splits / for up to two: hidden 4096, inter 14336, 32 rows K3 417.5 / 419.8 / 411.3, K4 422.7 / 429.2 / 417.4, 48
//     rows K4 538.9 / 534.1 / 525.4; inter 7168, 48 rows K4 431.2 / 428.0 / 428.1; hidden 5120, inter 13824, 32 rows K4 482.5 /
//     492.9 / 483.9; hidden 1024, inter 14336, 64 rows K5 385.8 / 394.9 (small grids at any K) / 387.4.
// Beyond 64 rows its loads of the activations bound it (64 KB per step and compute unit at 128 rows, 70 GB/s; 97 rows of
// 14336x4096 at K5 32.6 / 33.9); up to 16 rows half of its matrix instructions would be empty.
inline bool tile_takes(int K, int M, int S, int cb, int wgs) {
  if (M < 17 || M > 64) return false;
  const int cus = num_cu();
  if (S == 1 && wgs > cus) return M > 32 || K <= 4 || cb <= 16;
  return K <= 4 && cb >= 14 && S <= 2;
}
inline size_t batch_prerot_rows(int M, bool tile) { return tile ? (size_t)(M + 31) / 32 * 32 : (size_t)M; }   // rows the layout holds
inline size_t batch_lds_bytes(int M, bool tile) {
  if (tile) return tile_lds_bytes((M + 31) / 32);
  const int rows = 16 * batch_groups(M);
  const size_t blocks = (size_t)2 * rows * BATCH_ROWH * 2, small = (size_t)5 * rows * 4, fin = (size_t)2 * M * BATCH_FIN_STRIDE * 4;
  return M > 64 ? (blocks + small > fin ? blocks + small : fin) : blocks + small + fin;
}
// HTR_BATCH_ROT=0 switches the rotation by the workgroups off
inline bool batch_rot_on() {
  static const bool on = getenv("HTR_BATCH_ROT") == nullptr || atoi(getenv("HTR_BATCH_ROT")) != 0;
  return on;
}
// Who rotates a call's activations x: 0 a launch of its own, else the workgroups, as k_linear_batch's ROT says; 16-bit rows on 16-byte
// boundaries only
inline int batch_rot(int K, int M, int x_dtype, const void* x, const BatchPlan& bp) {
  if (x_dtype == HTR_F32 || ((uintptr_t)x & 15)) return 0;
  return bp.rot ? 1 : batch_rot_on() && batch_rot_long(K, M, bp.S, bp.cb, bp.wgs) ? 2 : 0;
}
inline size_t batch_rot_lds_bytes(int M, int cb, int rot) {
  const int rows = 16 * batch_groups(M);
  return (size_t)cb * rows * BATCH_ROWH * 2 + (size_t)cb * 2 * rows * 4 + rows * 4 +
         (rot == 1 ? (size_t)2 * M * BATCH_FIN_STRIDE * 4 : (size_t)cb * rows * 4);
}
inline bool make_batch_plan(int m, int n, int K, int M, int want_S, BatchPlan& bp) {
  const int nblk = n / 128, rbs = m / 128;
  if ((long)M * n * 2 >= (1L << 31)) return false;          // the kernels address the rotated activations with 32-bit byte offsets
  bp.mb = batch_groups(M);
  bp.rot = 0;
  // Measured on MI355X (K4, 6..128 rows, 1024..28672 output rows): one workgroup per CU is the best fill; every further
  // split adds partial traffic that grows with the rows (14336x4096, 32 rows: 2 splits 19.9 us, 4 splits 24.5; 128
  // rows: 39 against 48).  So: the largest split that keeps the grid within the CU count, among the splits that leave
  // no column range empty, and at most 8 of them (the output side requests the slots of up to eight other splits in
  // one go; 1024x4096 and 2048x4096 at 8..32 rows: 8 splits 11..12 us, 16 splits 11..16, 32 splits 14..22).
  const int cus = num_cu();
  const int by_cus = cus / rbs > 1 ? cus / rbs : 1;
  const int limit = want_S > 0 ? want_S : (by_cus < 8 ? by_cus : 8);
  bool found = false;
  for (int S = 1; S <= nblk && S <= limit; ++S) {
    const int cb = (nblk + S - 1) / S;
    if ((nblk + cb - 1) / cb != S) continue;                       // some split would be empty
    if (want_S > 0 && S != want_S) continue;
    bp.S = S; bp.cb = cb; bp.wgs = rbs * S; found = true;
  }
  if (!found) return false;
  bp.tile = tile_takes(K, M, bp.S, bp.cb, bp.wgs);
  if (bp.tile) {
    // The order for k_linear_tile has room for whole tiles of 32 rows, up to twice what the rows take.  What fits the library's
    // own workspace (htr_linear_static) as rows goes on fitting it, with k_linear_batch; and 32-bit offsets bound it as well.
    // (An order without gaps, offsets from the rows of the last tile, costs every call 0.2 to 0.4 us: 28672x4096, 64 rows K4 35.1 / 35.6.)
    const size_t slots = (size_t)bp.wgs * M * 128 * sizeof(float), padded = batch_prerot_rows(M, true);
    if ((padded * n * 2 >> 31) != 0 || (ws_need(slots, prerot_bytes(n, padded)) > HTR_STATIC_SCRATCH_BYTES &&
                                        ws_need(slots, prerot_bytes(n, M)) <= HTR_STATIC_SCRATCH_BYTES)) bp.tile = false;
  }
  bp.lds = batch_lds_bytes(M, bp.tile);
  // Splits that finish rows for each other wait for each other, which is only safe while every workgroup of the grid is
  // resident at once: one workgroup per CU at most.  A larger grid (an explicit split, a device with fewer CUs than the
  // policy assumed) falls back to the last split finishing everything: it waits only for workgroups dispatched before it.
  bp.last_finishes = bp.wgs > cus ? 1 : 0;
  // Few rows over few column blocks per split, one workgroup per CU: every workgroup rotates its own slice.
  if (batch_rot_on() && batch_rot_fits(M, bp.cb) && bp.wgs <= cus) {
    bp.rot = 1;
    bp.lds = batch_rot_lds_bytes(M, bp.cb, 1);
  }
  return true;
}

// ---- GEMM kernel (more than 128 rows): tiles of GEMM_ROWS activation rows in the grid's z, split S of the column blocks
// while the grid stays within one workgroup per compute unit (256 registers per lane leave room for one)
struct GemmPlan { int S, cb, mtiles, wgs, jb; };
constexpr int GEMM_MIN_M = HTR_MAX_ROWS_PER_TILE + 1;       // rows from which the library policy takes the GEMM kernel
inline bool gemm_plan_for(int m, int n, int M, int want_S, int jb, GemmPlan& gp) {
  const int nblk = n / 128, rbs = m / 128, rows = 32 * jb;
  if ((long)M * n * 2 >= (1L << 31)) return false;          // the kernel addresses the rotated activations with 32-bit byte offsets
  gp.jb = jb;
  gp.mtiles = (M + rows - 1) / rows;
  if (gp.mtiles > 65535) return false;
  const long base = (long)rbs * gp.mtiles;
  const int cus = num_cu();
  const int by_cus = cus / base > 1 ? (int)(cus / base) : 1;
  const int limit = want_S > 0 ? want_S : (by_cus < 4 ? by_cus : 4);
  bool found = false;
  for (int S = 1; S <= nblk && S <= limit && S <= 8; ++S) {
    const int cb = (nblk + S - 1) / S;
    if ((nblk + cb - 1) / cb != S) continue;                       // some split would be empty
    if (want_S > 0 && S != want_S) continue;
    gp.S = S; gp.cb = cb; gp.wgs = (int)(base * S); found = true;
  }
  return found;
}
// Tile height by a cost model in microseconds fitted to MI355X (K4): rounds of workgroups over the CUs x (steps per
// workgroup x 0.94 us with 96-row tiles, 1.16 us with 128-row tiles, + 10 us of fixed cost, + 4 + 1.5 (S - 1) us for the
// exchange between S column splits).  128-row tiles win where they save a round (14336x4096 at 256 rows: two tiles
// fill the chip once, 49 us, where three tiles of 96 rows take 73) or allow more splits of long rows (4096x14336 at 256
// rows: 55 against 64); 96-row tiles win otherwise (14336x4096 at 192 rows: 40 against 47; at 384 rows: 79 against 94).
// want_jb: 0 = this policy, 3 or 4 = that tile height.  By policy at most four splits (eight cost more than they save).
inline double gemm_plan_cost(const GemmPlan& gp) {
  const int cus = num_cu();
  const int rounds = (gp.wgs + cus - 1) / cus;
  return rounds * (gp.cb * (gp.jb == 3 ? 0.94 : 1.16) + 10.0 + (gp.S > 1 ? 4.0 + 1.5 * (gp.S - 1) : 0.0));
}
inline bool make_gemm_plan(int m, int n, int M, int want_S, int want_jb, GemmPlan& gp) {
  if (want_jb == 3 || want_jb == 4) return gemm_plan_for(m, n, M, want_S, want_jb, gp);
  GemmPlan a, b;
  const bool oka = gemm_plan_for(m, n, M, want_S, 3, a), okb = gemm_plan_for(m, n, M, want_S, 4, b);
  if (!oka && !okb) return false;
  gp = oka && (!okb || gemm_plan_cost(a) <= gemm_plan_cost(b)) ? a : b;
  return true;
}
// workspace of the GEMM kernel: one flag word per workgroup in the zeroed half; rotated activations and the exchange tiles
// (only with column splits) in the scratch half
inline size_t gemm_scratch_bytes(int n, int M, const GemmPlan& gp) {
  return prerot_bytes(n, M) + (gp.S > 1 ? (size_t)gp.wgs * (32 * gp.jb) * 128 * sizeof(float) : 0);
}
// nsplit bits 20 and 21 with the GEMM kernel: tiles of 96 or of 128 activation rows (neither: the policy above)
inline int gemm_want_jb(int nsplit) { return nsplit > 0 ? ((nsplit >> 20) & 1 ? 3 : ((nsplit >> 21) & 1 ? 4 : 0)) : 0; }
// nsplit bit 28: the GEMM kernel with the split in the low bits (0 = its own policy); otherwise from GEMM_MIN_M rows
inline bool wants_gemm(int M, int nsplit) { return nsplit > 0 ? (nsplit & (1 << 28)) != 0 : M >= GEMM_MIN_M; }

// ---- wide kernel: tiles of 256 activation rows, every tile's column blocks in S splits, the last tile's, which may hold fewer rows,
// in S_last, while the grid stays within one workgroup per compute unit
struct WidePlan { int S, S_last, cb, mtiles, wgs; };
constexpr int WIDE_MAX_SPLITS = 8;
inline bool split_fits(int nblk, int S) { const int cb = (nblk + S - 1) / S; return S >= 1 && S <= nblk && (nblk + cb - 1) / cb == S; }      // none empty
// For the choice of splits alone (wide_us says what a call takes): us per column block of a workgroup whose tile holds `rows` rows.  K4, 48
// workgroups on the chip: 96 rows 0.76, 128 rows 0.78, 256 rows 1.2 (from 129 rows on two waves of a SIMD multiply); exchange between S
// splits at 128 / 256 rows: 2 / 4.7 for two, 3 / 6.2 for four.  On 405 sizes at K 2 to 8 the chosen split takes 1.3 % more than the best
// one on average.  Five and seven splits are not among them: us at 4 / 5 / 6 / 7 of them, K4, 4096x4480 97 rows 21.9 / 21.6 / 20.9 / 23.6,
// 256 rows 32.3 / 34.5 / 33.3 / 37.4, 6144x8960 200 rows 48.8 / 47.3 / - / -, 256 rows 53.6 / 53.0 / - / -.
inline double wide_step_us(int rows) { return rows <= 128 ? 0.65 + 0.001 * rows : 0.96 + 0.001 * rows; }
inline double wide_exchange_us(int rows, int S) { return S == 1 ? 0.0 : (1.0 + 0.25 * S) * (rows <= 128 ? 1.0 : 2.0); }
inline bool make_wide_plan(int m, int n, int M, int want_S, WidePlan& wp) {
  const int nblk = n / 128, rbs = m / 128, cus = num_cu();
  if ((long)M * n * 2 >= (1L << 31)) return false;          // 32-bit byte offsets into the rotated activations; none beyond M n 2
  wp.mtiles = (M + WIDE_ROWS - 1) / WIDE_ROWS;
  const int rest = M - (wp.mtiles - 1) * WIDE_ROWS;
  if ((long)rbs * wp.mtiles * WIDE_MAX_SPLITS >= (1L << 31)) return false;
  double best = 1e30;
  for (int S = 1; S <= WIDE_MAX_SPLITS; ++S) {
    if (!split_fits(nblk, S) || (want_S > 0 ? S != want_S : S == 5 || S == 7)) continue;
    for (int L = 1; L <= WIDE_MAX_SPLITS; ++L) {
      if (!split_fits(nblk, L) || (want_S > 0 ? L != want_S : L == 5 || L == 7) || (wp.mtiles == 1 && L != S)) continue;
      const long wgs = (long)rbs * (S * (long)(wp.mtiles - 1) + L);
      const long rounds = (wgs + cus - 1) / cus;
      if (want_S == 0 && rounds > 1 && S + L > 2) continue;
      const double full = wp.mtiles > 1 ? ((nblk + S - 1) / S) * wide_step_us(WIDE_ROWS) + wide_exchange_us(WIDE_ROWS, S) : 0.0;
      const double part = ((nblk + L - 1) / L) * wide_step_us(rest) + wide_exchange_us(rest, L);
      const double cost = rounds * (full > part ? full : part) + (S != L ? 2.0 : 0.0);
      if (cost < best) { best = cost; wp.S = S; wp.S_last = L; wp.cb = (nblk + S - 1) / S; wp.wgs = (int)wgs; }
    }
  }
  return best < 1e30;
}
// partial slots of all splits: [workgroup][rows of its tile][128] floats (the last tile's workgroups come last)
inline size_t wide_slot_bytes(int m, int M, const WidePlan& wp) {
  if (wp.S == 1 && wp.S_last == 1) return 0;
  const size_t full = (size_t)(wp.mtiles - 1) * (m / 128) * wp.S * WIDE_ROWS, rest = (size_t)(m / 128) * wp.S_last * (M - (wp.mtiles - 1) * WIDE_ROWS);
  return (full + rest) * 128 * sizeof(float);
}
// The wide kernel: nsplit bit 27, with the split of all tiles in the low bits (0 = its own policy), and by policy from 65 rows to 128.
// us of the call with its rotation, in a graph over several weights, k_linear_batch / k_linear_wide: 14336x4096 K4 65 rows 32.6 / 26.9, 97
// rows 35.2 / 32.1, 128 rows 38.0 / 33.7, K8 97 rows 39.3 / 33.1, K5 float16 97 rows 36.5 / 30.6; 4096x14336 K4 65 rows 32.8 / 28.9, K8
// 128 rows 41.7 / 40.7; 2048x2048 K4 128 rows 17.1 / 15.5; 28672x4096 K4 128 rows 61.3 / 48.8.  Of 260 sizes (13 matrices, K 2 to 8, 65
// to 128 rows) it was behind in none; the nearest, 1024x1024 K5 65 rows, 13.3 / 13.1 and, measured again, 12.6 / 12.8.  At 64 rows it is
// behind (14336x4096 K4 23.9 / 25.7, 2048x2048 11.9 / 13.1).  From 129 rows against k_linear_gemm: 6144x4096 K4 129 rows 32.2 / 24.3, 256
// rows 40.1 / 29.7, 333 rows 39.8 / 37.1; 14336x4096 256 rows 50.6 / 44.3, 333 rows 76.3 / 60.4, 512 rows 94.9 / 72.4; 4096x14336 256 rows
// 60.6 / 52.2 (htr_linear_route says who takes it there).
constexpr int WIDE_MIN_M = 65, NSPLIT_WIDE = 1 << 27;
inline bool wants_wide(int M, int nsplit) {
  return nsplit > 0 ? (nsplit & NSPLIT_WIDE) != 0 : M >= WIDE_MIN_M && M <= HTR_MAX_ROWS_PER_TILE;
}
inline int wide_want_S(int nsplit) { return nsplit > 0 ? nsplit & 0xFFFFF : 0; }

// Rows up to which a matrix is always multiplied by a fused launch, the wide kernel's: the codes stay exact there (2e-4 against float64,
// 2.4e-3 with a dequantized weight, whose entries are bfloat16).  The other kernel for these rows, k_linear_gemm, is no further choice:
// of 476 shapes within them (K 2 to 8, 129 to 512 rows, GPU time) it was ahead in three, and measured again in one (10240x2560 K3 245
// rows, 33.5 / 34.6 us; 4096x4096 K8 192 and 256 rows 33.4 / 27.6, 39.3 / 35.5); it took 1.03 to 1.76 times the wide kernel's time in
// the others.  Dequantization and product was ahead of the wide kernel in none of 276 (4096x4096 K8 256 rows 37.1).
// Beyond these rows float32 activations stay float32: the fused kernels round the rotated activations to float16, which only the
// library's product on the dequantized weight does not.
inline int fused_rows(int m, int n) {
  return (long)m * n < 4096L * 4096 ? HTR_MAX_ROWS_PER_TILE : n >= 8192 ? 512 : 384;
}

// Beyond fused_rows: the wide kernel, or the weight dequantized and the library's product?  Two models in us of GPU time, fitted to 2394
// measurements (256x256 to 28672x14336 and the matrices of common models, 129 to 2048 rows, K 2 to 8, bfloat16 and float16) and sweeps of
// splits.  The wide kernel's is within 8 % for nine in ten.  The library's product varies by more from one size to the next; its model is
// fitted so that two calls in five are faster, and the wide kernel is taken where it is 4 % ahead of that.  Of 975 sizes that were not
// fitted it is taken for 366 in a graph and more than 3 % behind in seven (of 800 queued eagerly for 526, and eight), 29 % at worst
// (4352x384 K5 1913 rows float16 36 / 28); for 77 (66) that are dequantized it would be more than 3 % ahead.  Wide / dequantized, us
// in a graph, K4 and bfloat16 where nothing else is said: 14336x4096 512 rows 80 / 99, 1024 rows 149 / 144, K8 156 / 142; 3072x3072 333
// rows 27 / 36; 2048x2048 200 rows 19.7 / 18.1; 10624x8320 934 rows 235 / 200; 6400x512 K8 171 rows 18.3 / 16.3; 24448x3712 K8 584 rows
// float16 146 / 362.
//
// Time of a grid of `full` workgroups of t_full us and, behind them, `last` ones of t_last us: they start in order, each on the compute
// unit that is free first, so short ones fill the places beside a round of full ones that does not take all units.
inline double grid_us(long full, double t_full, long last, double t_last, int cus) {
  const long early = cus - full % cus, late = full % cus;             // units that do one full workgroup less, and the others
  double t_early = (double)(full / cus) * t_full, t_late = t_early + t_full, end = late > 0 ? t_late : t_early;
  while (last > 0) {
    const bool on_early = late == 0 || t_early <= t_late;
    double& t = on_early ? t_early : t_late;
    last -= on_early ? early : late;
    t += t_last;
    if (t > end) end = t;
  }
  return end;
}
// Launches; rotation; the workgroups, each with first loads and decode, steps that take longer with more bits, and an output side by
// its rows; partials of column splits by their bytes (written, read, cleared); output; and the matrix work of the whole chip, which slows
// all steps the more of it there is.
inline double wide_us(int m, int n, int K, int M, const WidePlan& wp) {
  const int nblk = n / 128, rest = M - (wp.mtiles - 1) * WIDE_ROWS;
  const long full = (long)(m / 128) * wp.S * (wp.mtiles - 1), last = (long)(m / 128) * wp.S_last;
  auto workgroup = [&](int rows, int S) {
    const double step = rows <= 128 ? 0.68 + 0.0007 * rows + 0.02 * (K - 4) : 1.05 + 0.025 * (K - 4);
    return 4.7 + ((nblk + S - 1) / S) * step + 0.025 * rows;
  };
  const double partials = 512.0 * ((wp.S > 1 ? (double)full * WIDE_ROWS : 0.0) + (wp.S_last > 1 ? (double)last * rest : 0.0));
  return 4.6 + 2.1e-6 * M * n + grid_us(full, workgroup(WIDE_ROWS, wp.S), last, workgroup(rest, wp.S_last), num_cu()) + 0.14e-6 * partials +
         0.15e-6 * M * m + 0.68e-9 * M * m * n;
}
// Launches; dequantization; product, its output, and a serial part by columns, which is less for few tiles (of 128x128: the library then
// splits the columns) and comes again with every round of 256x256 tiles over the chip; float16 converts the weight once more.
inline double dequant_us(int m, int n, int M, int x_dtype) {
  const double weights = (double)m * n;
  const int cus = num_cu();
  const long few = (long)(m / 128) * ((M + 127) / 128), tiles = (long)((m + 255) / 256) * ((M + 255) / 256), rounds = (tiles + cus - 1) / cus;
  const double columns = 1.22e-3 * n * (few < 50 ? few / 50.0 : 1.0) + 1.37e-3 * n * rounds;
  return 9.7 + weights * 0.86e-6 + M * weights * 0.99e-9 + 1.17e-6 * M * m + columns + (x_dtype == HTR_BF16 ? 0.0 : 3.5 + weights * 1.6e-6);
}
// eager: the call is queued by itself.  The host then takes 23 to 25 us for dequantization and product (28 to 30 with the conversion), and
// 9 for a wide launch; longer calls take what the GPU takes.
inline bool wide_ahead(int m, int n, int K, int M, int x_dtype, const WidePlan& wp, bool eager) {
  double wide = wide_us(m, n, K, M, wp), dequant = dequant_us(m, n, M, x_dtype);
  if (eager) {
    const double host = x_dtype == HTR_BF16 ? 23.5 : 28.5;
    if (wide < 9.0) wide = 9.0;
    if (dequant < host) dequant = host;
  }
  return 1.04 * wide < dequant;
}

struct BatchArgs { const uint32_t* qw; float* part; const void* x; const uint8_t* su; int m, n, M, flags; };
template <int K, int MB, int ROT> int launch_batch_v(const BatchArgs& a, const LinearTail& t, const BatchPlan& bp, hipStream_t st) {
  const size_t lds = balanced_lds_request(bp.lds, bp.wgs);
  HTR_CHECK_HIP((allow_full_lds<k_linear_batch<K, MB, 4, ROT>>()));
  HTR_CHECK_HIP(launch_kernel(k_linear_batch<K, MB, 4, ROT>, dim3(bp.S, a.m / 128), dim3(WG_THREADS), lds, st, a.qw, a.part, a.x, a.su,
                              a.m, a.n, a.M, bp.S, a.flags, t));
  return HTR_OK;
}
// ONE: one split, an instantiation without the exchange between splits: few enough registers (128) for two workgroups per
// compute unit also with two row tiles, where one workgroup's decode covers the other's first loads and output side.  The
// second workgroup replaces the deeper rings: two stream buffers and one set of fragments instead of four and two.
template <int K, int JB, bool ONE> int launch_tile_v(const BatchArgs& a, const LinearTail& t, int S, int problems, hipStream_t st) {
  constexpr int P = K > 4 || (ONE && JB > 1) ? 2 : 4, DB = ONE && JB > 1 ? 1 : 2;
  const size_t lds = problems == 1 || !ONE ? balanced_lds_request(tile_lds_bytes(JB), S * (a.m / 128) * problems) : tile_lds_bytes(JB);
  HTR_CHECK_HIP((allow_full_lds<k_linear_tile<K, JB, P, DB, ONE>>()));
  HTR_CHECK_HIP(launch_kernel(k_linear_tile<K, JB, P, DB, ONE>, dim3(S, a.m / 128, problems), dim3(WG_THREADS), lds, st, a.qw, a.part, a.m, a.n,
                              a.M, S, a.flags, t));
  return HTR_OK;
}
template <int K> int launch_wide_k(const BatchArgs& a, const LinearTail& t, const WidePlan& wp, hipStream_t st) {
  HTR_CHECK_HIP((allow_full_lds<k_linear_wide<K>>()));
  HTR_CHECK_HIP(launch_kernel(k_linear_wide<K>, dim3(wp.wgs), dim3(WG_THREADS), WIDE_LDS, st, a.qw, a.part, a.m, a.n, a.M, wp.S, wp.S_last, a.flags, t));
  return HTR_OK;
}
// Grouped launches of 9 to 32 rows per problem: column splits while every workgroup of the grid has a compute unit to itself, as
// for one linear (make_batch_plan); the splits of a row block wait for each other.  Measured on MI355X, K4, us, chunked kernel /
// k_linear_tile without splits / with, rotation included: one problem of 4096x14336 with 9 rows 32.3 / 55.8 / 17.9, with 32 rows
// 72.2 / 60.0 / 20.6; two of 256x4096 with 9 rows 16.2 / 21.1 / 11.6; two of 1024x1024 with 9 rows 10.9 / 11.3 / 10.3.
inline int group_tile_splits(int count, int m, int n) {
  const int nblk = n / 128, limit = num_cu() / count / (m / 128);
  int best = 1;
  for (int S = 2; S <= nblk && S <= limit && S <= 8; ++S) {
    const int cb = (nblk + S - 1) / S;
    if ((nblk + cb - 1) / cb == S) best = S;                       // no split is empty
  }
  return best;
}
// Whether k_linear_tile takes the group.  The chunked kernel keeps up to 8 rows (not compared) and, at five bits and more, up to
// 12 rows of problems with long rows whose row blocks leave a quarter of the last round over the compute units empty, which its
// chunks fill.  us, chunked / k_linear_tile: twelve problems of 4096x4096 with 9 rows K4 41.5 / 40.3, K5 44.0 / 50.3, K8 54.6 / 57.7,
// with 16 rows K5 65.1 / 51.3; twelve of 4096x14336 with 9 rows K4 124 / 120, K5 137 / 158; six of them K5 77.9 / 84.4, eight
// 99.2 / 91.1; six of 4096x4096 K5 31.9 / 28.3; twelve of 2816x2048 K5 34.4 / 26.8.  (Left as they are: ten of 4096x14336 or
// 4096x8192 with 9 rows at K4, 7 % behind the chunked kernel.)
inline bool group_takes_tiles(int count, int m, int n, int K, int max_M) {
  if (max_M <= 8) return false;
  if (K <= 4 || max_M > 12 || group_tile_splits(count, m, n) > 1) return true;
  const int nblk = n / 128, cus = num_cu(), grid = count * (m / 128), rounds = (grid + cus - 1) / cus;
  return rounds > 2 || nblk < (rounds == 1 ? 64 : 32) || 4 * grid > 3 * rounds * cus;
}
template <int K> int launch_batch_k(const BatchArgs& a, int rot, const LinearTail& t, const BatchPlan& bp, hipStream_t st) {
  if (rot == 1) return bp.mb == 1 ? launch_batch_v<K, 1, 1>(a, t, bp, st) : launch_batch_v<K, 2, 1>(a, t, bp, st);
  if (rot == 2) return bp.mb == 1 ? launch_batch_v<K, 1, 2>(a, t, bp, st) : launch_batch_v<K, 2, 2>(a, t, bp, st);
  if (bp.tile) {
    // Grids beyond one workgroup per compute unit, us without / with ONE: K4, 64 rows 65536x4096 67.0 / 59.4, 40960x1024 28.7 /
    // 22.4, 33 rows 152064x4096 137.6 / 115.9; 17 rows 40960x2048 24.0 / 23.6, 32 rows 25.5 / 24.7, 65536x4096 45.4 / 44.9.  Up to one
    // per unit there is no second workgroup to gain from: eight decoder layers of 32 rows at K3, whose gate/up takes 224 workgroups, 558 to 562 / 565 to 571.
    const bool one = bp.S == 1 && bp.wgs > num_cu();
    if (one) return a.M <= 32 ? launch_tile_v<K, 1, true>(a, t, 1, 1, st) : launch_tile_v<K, 2, true>(a, t, 1, 1, st);
    if constexpr (K <= 4) return a.M <= 32 ? launch_tile_v<K, 1, false>(a, t, bp.S, 1, st) : launch_tile_v<K, 2, false>(a, t, bp.S, 1, st);
  }
  switch (bp.mb) {
    case 1: return launch_batch_v<K, 1, 0>(a, t, bp, st);
    case 2: return launch_batch_v<K, 2, 0>(a, t, bp, st);
    case 4: return launch_batch_v<K, 4, 0>(a, t, bp, st);
    default: return launch_batch_v<K, 8, 0>(a, t, bp, st);
  }
}
// nsplit bit 29: batched kernel with the split in the low bits (0 = policy); otherwise the policy decides by M
// Tall matrices (192 row blocks and more) fill the chip without column splits, so the batched kernel needs no exchange
// there and wins from 6 rows (65536x4096, 8 rows: 41 against 50 us; 152064x4096: 91 against 95).
// A matrix whose splits are four column blocks or fewer on a full grid (4096x4096: 8 splits of 4 blocks) is also ahead
// with the batched kernel at 7 and 8 rows, when its workgroups rotate their own slices (8 rows: 9.2 against 10.4 us).
inline bool wants_batch(int M, int nsplit, int m, int n, int K) {
  if (wants_gemm(M, nsplit)) return false;
  if (nsplit > 0) return (nsplit & (1 << 29)) != 0;
  if (M >= BATCH_MIN_M || (M >= 6 && m / 128 >= 192)) return true;
  if (M >= 7) {
    BatchPlan bp;
    return make_batch_plan(m, n, K, M, 0, bp) && bp.rot && bp.cb <= 4 && bp.wgs >= num_cu();
  }
  return false;
}

// Rotation of all rows of x ahead of a linear launch: on the matrix unit for 16-bit rows on 16-byte boundaries, else the
// butterfly kernel (float32, odd alignments)
// (frag: not 0 = in fragment order for that many rows, FRAG_FULL = in whole tiles)
inline hipError_t launch_rotation(const void* x, const uint8_t* su, int n, int M, int x_dtype, const LinearTail& t, hipStream_t st, size_t frag = 0) {
  static const bool mfma_on = getenv("HTR_ROTATE_MFMA") == nullptr || atoi(getenv("HTR_ROTATE_MFMA")) != 0;
  if (mfma_on && x_dtype != HTR_F32 && ((uintptr_t)x & 15) == 0)
    return launch_kernel(k_rotate_mfma, dim3((n / 128 + 4 * WG_WAVES - 1) / (4 * WG_WAVES), M), dim3(WG_THREADS), 0, st, x, su, n,
                         x_dtype == HTR_BF16 ? 1 : 0, (_Float16*)t.xt_g, (float*)t.xs_g, (float*)t.sc_g, frag);
  return launch_kernel(k_rotate, dim3((n / 128 + WG_WAVES - 1) / WG_WAVES, M), dim3(WG_THREADS), 0, st, x, su, n, x_dtype,
                       (_Float16*)t.xt_g, (float*)t.xs_g, (float*)t.sc_g, (const htr_group_entry*)nullptr, 0ull, frag);
}

#define HTR_FOR_K_OR(K, EXPR, OTHERWISE)   \
  switch (K) {                             \
    case 2: { constexpr int KK = 2; EXPR; } break; \
    case 3: { constexpr int KK = 3; EXPR; } break; \
    case 4: { constexpr int KK = 4; EXPR; } break; \
    case 5: { constexpr int KK = 5; EXPR; } break; \
    case 6: { constexpr int KK = 6; EXPR; } break; \
    case 7: { constexpr int KK = 7; EXPR; } break; \
    case 8: { constexpr int KK = 8; EXPR; } break; \
    default: OTHERWISE;                    \
  }
#define HTR_FOR_K(K, EXPR) HTR_FOR_K_OR(K, EXPR, return HTR_ERR_K)

inline bool dtype_ok(int d) { return d == HTR_BF16 || d == HTR_F16 || d == HTR_F32; }

