// C ABI of libonebitmul (declared in include/onebit_sparse_tensor.h): argument validation, per-device
// workspaces, kernel selection. Host code only; the kernels live in onebit_gemm*, onebit_skinny*, onebit_wide* and
// onebit_format.hip.
// Counterpart of the reference's host launcher csrc/kernel_lib.cu:23-97.
#include "onebit_sparse_tuning.h"
#include "onebit_device.h"
#include "onebit_launch.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

thread_local std::string g_last_error;
// Tuning / test hooks: per calling thread, so that a test or a tuning run never changes what other threads of the
// process launch.
thread_local int g_tile_config = -1;
thread_local int g_skinny_enabled = 1;
thread_local int g_skinny_rows = -1;
thread_local int g_split_k = -1;
thread_local int g_pad_b = 1;
std::atomic<int> g_weight_cache_entries{0};

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

#define ONEBIT_HIP(expr)                                                                         \
  do {                                                                                           \
    hipError_t st_ = (expr);                                                                     \
    if (st_ != hipSuccess)                                                                       \
      return fail(ONEBIT_ERR_HIP, "HIP error '%s' from %s", hipGetErrorString(st_), #expr);      \
  } while (0)

constexpr int kMaxDevices = 64;

// Workspace of onebit_sparse_matmul_prepared_static: device memory that exists from the moment the code object is
// loaded, so that entry point never allocates. Every GPU the library runs on holds its own copy at its own address
// until the process ends. In host code the name is only a handle for hipGetSymbolAddress; kernels and copies use the
// per-device address kept in DeviceState::static_scratch.
constexpr size_t kStaticScratchBytes = ONEBIT_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char g_static_scratch[kStaticScratchBytes];

// Library-owned device memory. Grow-only, one buffer per device and stream (calls on one stream are ordered, calls
// on different streams must not share a buffer), freed at process exit by the runtime.
struct Buffer {
  void* ptr = nullptr;
  size_t bytes = 0;
};
struct DeviceState {
  // recursive: the one-call entry points keep it while they launch, and the launch takes it again for its own buffers
  std::recursive_mutex mu;
  // the reordered operand of the one-call entry points (when the weight cache is off)
  std::map<hipStream_t, Buffer> prep;
  // fp32 partial sums of the K-split passes: one buffer per stream, so that calls on different streams do not
  // share one (calls on the same stream are ordered)
  std::map<hipStream_t, Buffer> split_ws;
  // B with rows padded to a multiple of 8 columns (operands the asynchronous copies cannot read in place), per stream
  std::map<hipStream_t, Buffer> b_pad;
  // opt-in cache of prepared operands of the one-call entry points, keyed by the caller's weight pointers
  struct CachedWeight {
    const void* a;
    const void* e;
    int m, k, layout;
    void* prep;
    hipStream_t stream;  // the stream its reorder kernel was enqueued on
    hipEvent_t ready;    // recorded after that kernel
    unsigned long last_use;
  };
  std::vector<CachedWeight> weight_cache;
  unsigned long use_counter = 0;
  // compute units of the device (0 until first asked): the launch plans scale with it
  std::atomic<int> compute_units{0};
  // this device's address of g_static_scratch (null until the first non-allocating call on the device)
  unsigned char* static_scratch = nullptr;
};
DeviceState g_dev[kMaxDevices];

// Grows a library-owned buffer. Growing frees the old memory after a device synchronization: a HIP graph captured
// earlier on this stream still holds the old address and must be captured again after a larger call. Inside a stream
// capture neither the synchronization nor the allocation is possible, so a call that would have to grow there is
// refused instead of invalidating the capture. `reserve`: size to grow to, at least `need`, where that is possible.
int grow(void** ptr, size_t* have, size_t need, hipStream_t stream, size_t reserve = 0) {
  reserve = std::max(need, reserve);
  if (reserve <= *have) return ONEBIT_OK;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  ONEBIT_HIP(hipStreamIsCapturing(stream, &capture));
  if (capture != hipStreamCaptureStatusNone) {
    if (need <= *have) return ONEBIT_OK;
    return fail(ONEBIT_ERR_ARGUMENT,
                "a library-owned buffer would have to grow to %zu bytes while the stream is being captured: run the "
                "call once outside the capture first, or use the non-allocating entry point", need);
  }
  if (*ptr) {
    // earlier work on any stream may still read the old buffer
    ONEBIT_HIP(hipDeviceSynchronize());
    ONEBIT_HIP(hipFree(*ptr));
    *ptr = nullptr;
    *have = 0;
  }
  const size_t bytes = (reserve + 4095) & ~size_t(4095);
  ONEBIT_HIP(hipMalloc(ptr, bytes));
  *have = bytes;
  return ONEBIT_OK;
}

// Compute units of the current device, asked once per device. A failure leaves the MI355X figure the plans were
// measured on.
int current_compute_units() {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return 256;
  int cus = g_dev[device].compute_units.load(std::memory_order_relaxed);
  if (cus > 0) return cus;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0) cus = 256;
  g_dev[device].compute_units.store(cus, std::memory_order_relaxed);
  return cus;
}

int check_shape(int m, int n, int k) {
  if (m <= 0 || n <= 0 || k <= 0) return fail(ONEBIT_ERR_ARGUMENT, "m, n, k must be positive (got %d, %d, %d)", m, n, k);
  if (m % 64 != 0) return fail(ONEBIT_ERR_ARGUMENT, "m = %d must be a multiple of 64 (metadata layout)", m);
  if (k % 32 != 0) return fail(ONEBIT_ERR_ARGUMENT, "k = %d must be a multiple of 32 (metadata layout)", k);
  return ONEBIT_OK;
}

int check_dtype(int c_dtype, int d_dtype) {
  if ((c_dtype != ONEBIT_DTYPE_F32 && c_dtype != ONEBIT_DTYPE_F16) ||
      (d_dtype != ONEBIT_DTYPE_F32 && d_dtype != ONEBIT_DTYPE_F16))
    return fail(ONEBIT_ERR_ARGUMENT, "dtype codes must be 0 (fp32) or 1 (fp16), got c=%d d=%d", c_dtype, d_dtype);
  return ONEBIT_OK;
}

// The linear layer's types: 16-bit activations, a result of their type or fp32, any bias.
int check_linear_dtypes(int x_dtype, int bias_dtype, int y_dtype) {
  if (x_dtype != ONEBIT_DTYPE_F16 && x_dtype != ONEBIT_DTYPE_BF16)
    return fail(ONEBIT_ERR_ARGUMENT, "x dtype code must be 1 (fp16) or 2 (bf16), got %d", x_dtype);
  if (y_dtype != ONEBIT_DTYPE_F32 && y_dtype != x_dtype)
    return fail(ONEBIT_ERR_ARGUMENT, "y dtype code must be 0 (fp32) or that of x (%d), got %d", x_dtype, y_dtype);
  if (bias_dtype < ONEBIT_DTYPE_F32 || bias_dtype > ONEBIT_DTYPE_BF16)
    return fail(ONEBIT_ERR_ARGUMENT, "bias dtype code must be 0 (fp32), 1 (fp16) or 2 (bf16), got %d", bias_dtype);
  return ONEBIT_OK;
}

// Tile and number of K splits of the main kernel. The time is rounds of resident workgroups times one workgroup's K
// loop; the choice among the tiles, and among splits of K that fill idle compute units at the price of a second launch
// and of writing and re-reading fp32 partial sums, comes from a cost model fitted to measurements on MI355X
// (microseconds):
//   K loop of one workgroup per 256-wide chunk with every slot of the GPU taken: 512 x 128: 3.8, 256 x 128 on eight
//   wavefronts: 2.3, on four (two workgroups per CU): 3.9, 128 x 128 on four (two per CU): 2.4, as two K groups:
//   1.2, as 64 x 32 wavefronts: 1.5, 64 x 128: 1.0, as two K groups: 0.88;
//   a round that fills only a fraction f of the slots is shorter: with one workgroup per CU 0.85 of a full round
//   below f = 0.9; with two per CU 0.6 up to f = 0.5 (every workgroup has its CU to itself) and a full round above
//   (some CUs hold two again); the two-K-group tiles pay 1.5 and 1.0 per round for exchanging the groups' sums;
//   4 for launch, prologue and epilogue; a split adds 5 and moves (S + 1) partial results at about 5 TB/s.
// Examples the model was checked against (measured, us): 4096 x 3072 x 4096: 512 x 128 57.0, 256 x 128 68.3;
// 4096 x 1536 x 4096: 256 x 128 35.0, 128 x 128 38.9; 4096 x 384 x 11008: 64 x 128 40.2, 256 x 128 with four splits
// 32.5; 11008 x 768 x 4096: 512 x 128 51.2, 256 x 128 65.5; 4096 x 128 x 4096: 64 x 128 with four splits 13.9,
// unsplit 17.3.
struct GemmPlan {
  int tile;
  int splits;
  double us;  // modelled; 0 for a forced tile
};

struct TileCost {
  int tile, bm, bn;
  int slots;        // workgroups resident at once on the 256 compute units the timings were taken on
  double chunk_us;  // K loop of one workgroup per 256-wide chunk with every slot taken
  double round_us;  // per round on top of the K loop
  bool may_split;
};
const TileCost kTileCosts[] = {
    {onebit::kTile512x128w8, 512, 128, 256, 3.8, 0.0, false}, {onebit::kTile256x128w8, 256, 128, 256, 2.3, 0.0, true},
    {onebit::kTile256x128w, 256, 128, 512, 3.9, 0.0, false},  {onebit::kTile128x128s, 128, 128, 512, 2.4, 0.0, false},
    {onebit::kTile128x128k2, 128, 128, 256, 1.2, 1.5, true}, {onebit::kTile128x128w8, 128, 128, 256, 1.5, 0.0, true},
    {onebit::kTile64x128, 64, 128, 256, 1.0, 0.0, true},      {onebit::kTile64x128k2, 64, 128, 256, 0.88, 1.0, true},
};

// compute_units: of the device the call runs on. The per-chunk times are per workgroup and do not depend on it; the
// number of resident workgroups scales with it (a partitioned or smaller GPU runs more rounds of the same tiles).
double model_us(const TileCost& t, int m, int n, int chunks, int s, int compute_units) {
  const long tiles = (long)((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn) * s;
  const int per_split = (chunks + s - 1) / s;
  const long slots = std::max(1L, (long)t.slots * compute_units / 256);
  const long full_rounds = tiles / slots;
  const double f = (double)(tiles % slots) / slots;
  double rounds = (double)full_rounds;
  if (f > 0.0) rounds += t.slots == 256 ? (f > 0.9 ? 1.0 : 0.85) : (f <= 0.5 ? 0.6 : 1.0);
  double us = 4.0 + (t.chunk_us * per_split + t.round_us) * rounds;
  if (s > 1) us += 5.0 + (s + 1) * 4.0 * m * n / 5.0e6;
  return us;
}

GemmPlan plan_gemm(int m, int n, int k, int compute_units) {
  const int chunks = (k + onebit::kChunkK - 1) / onebit::kChunkK;
  const int forced_tile = g_tile_config;
  const int forced_splits = g_split_k;
  if (forced_tile >= 0) {
    // a forced tile of the table may still be split by the model
    int splits = forced_splits >= 1 ? forced_splits : 1;
    if (forced_splits < 1)
      for (const TileCost& t : kTileCosts)
        if (t.tile == forced_tile && t.may_split) {
          double best_us = 1e30;
          for (int s : {1, 2, 3, 4, 6, 8, 12, 16}) {
            if (s > chunks) break;
            const double us = model_us(t, m, n, chunks, s, compute_units);
            if (us < best_us) best_us = us, splits = s;
          }
        }
    if (splits > chunks) splits = chunks;
    return GemmPlan{forced_tile, splits, 0.0};
  }
  const int fixed_splits = forced_splits >= 1 ? (forced_splits > chunks ? chunks : forced_splits) : 0;
  GemmPlan best{onebit::kTile128x128s, fixed_splits ? fixed_splits : 1, 0.0};
  double best_us = 1e30;
  auto consider = [&](const TileCost& t, int s) {
    const double us = model_us(t, m, n, chunks, s, compute_units);
    if (us < best_us) {
      best_us = us;
      best = GemmPlan{t.tile, s, us};
    }
  };
  for (const TileCost& t : kTileCosts) {
    if (fixed_splits) {
      consider(t, fixed_splits);
      continue;
    }
    for (int s : {1, 2, 3, 4, 6, 8, 12, 16}) {
      if (s > chunks || (s > 1 && !t.may_split)) break;
      consider(t, s);
    }
  }
  // With every compute unit busy the 512 x 128 tile is bound by power, and the same tile built on the 16x16x64 SMFMAC
  // (four wavefronts, one per SIMD) draws less of it per product: 3-5 % faster from about one full round of tiles on
  // (8192^3, 4096^3, 25600^3; 28672 x 512 x 8192 with 224 tiles: 102.9 against 107.0 us), slower when part of the chip
  // idles and the schedule decides (4096 x 3072 x 4096 with 192 tiles: 51.2 against 50.6; 11008 x 768 x 4096: 49 against 41).
  if (best.tile == onebit::kTile512x128w8 && best.splits == 1) {
    const long tiles = (long)((m + 511) / 512) * ((n + 127) / 128);
    // From 85 % of a round on; on K from 43 chunks on, where the epilogue of its four wavefronts weighs less, from three quarters on.
    // us, eight wavefronts | four (layers in fp16 with a bias, layers with fp32 results, products, products with fp32 C and results),
    // 192, 200 and 208 tiles: 4096 x 11008 with 3072 127 | 120, 129 | 126, 126 | 121, 138 | 136; 5120 x 11008 with 2560 131 | 123,
    // 133 | 129, 130 | 124, 142 | 139; 8192 x 16384 with 1600 194 | 183, 195 | 191, 193 | 186, 204 | 199. On shorter K the gain shrinks
    // with the chunks, for fp32 results first: from 34 chunks on all four forms are still equal or faster (34: 4096 x 8704 with 3072 103 |
    // 97, 104 | 103, 101 | 97, 115 | 114), at 32 fp32 results are equal (98.4 | 98.4, 109.2 | 109.6); the line is on the safe side.
    if (tiles * 20 >= 17L * compute_units || (chunks >= 43 && tiles * 4 >= 3L * compute_units)) best.tile = onebit::kTile512x128m16;
  }
  return best;
}

// Everything the C ABI decides about one prepared call, from the shape and the alignment of B alone (no GPU needed).
struct LaunchPlan {
  int split_k_kernel;  // 1: skinny_kernel, 0: gemm_kernel
  int rows_or_tile;    // skinny_kernel: weight rows per workgroup; gemm_kernel: TileConfig
  int splits;          // gemm_kernel: K splits over workgroups (1 = none)
  int pad_b;           // gemm_kernel: B is read through a padded copy
  double model_us;     // gemm_kernel: what the plan is modelled to take
};

// Row group and K splits over workgroups of the split-K kernel. Every workgroup of that kernel reads all of B's rows
// of its K range, so with few row groups over a long K (4096 x 28672 x 16: 128 workgroups that each read 900 KB of B
// for 170 KB of weights) the compute units spend their time re-reading B and half of them have no workgroup at all.
// Splitting K over S workgroups per row group divides both; the price is a second launch that adds the S partial
// results (about 3 us in all). Rule fitted to a sweep of m = 2048 ... 11008, k = 4096 ... 28672, n = 16, 32, 64 over
// every row group and S = 1 ... 8 (us, unsplit -> split): 2048 x 28672 x 16 18.5 -> 9.2, 4096 x 16384 x 16 12.0 -> 9.1,
// 4096 x 28672 x 32 28.0 -> 15.6, 8192 x 28672 x 16 21.4 -> 18.4, 8192 x 16384 x 64 30.2 -> 23.0, 11008 x 28672 x 32
// 34.2 -> 28.9; the best split always has at most one workgroup per compute unit and 64-row groups (128 rows when 64
// rows leave no room for two splits); below the threshold on B's bytes per workgroup the second launch costs more
// than the split saves (4096 x 11008 x 16: 8.9 against 8.5).
struct SkinnyPlan {
  int rows, splits;
};

// Weight rows per workgroup of the split-K kernel up to sixteen columns, from the workgroups that 32 and 64 rows give: the smallest
// whose workgroups have a compute unit each. A workgroup more than that waits for a second round (us, 32 | 64 | 128 rows, both forms
// alike: 9216 x 4096 with one token 6.0 | 4.6 | 6.6, with sixteen 7.3 | 5.4 | 7.2, with three columns 8.3 | 6.3 | 8.3; 17408 x
// 4096 9.4 | 8.5 | 7.0, 11.2 | 10.2 | 7.6, 12.4 | 11.8 | 8.8; 18432 x 8192 with sixteen 15.9 | 14.6 | 11.5; on short K 64 | 128
// rows: 18688 x 1280 with one / four columns, three / sixteen tokens 6.6 | 5.4, 5.3 | 5.3, 6.5 | 5.3, 7.7 | 6.1, x 512 5.4 | 4.2, 4.5 |
// 4.3, 5.4 | 4.2, 6.6 | 5.1), and a larger group
// leaves compute units idle (8192 x 4096 with one token 3.9 | 4.6 | 6.6, 16384 x 4096 7.3 | 5.4 | 7.0).
int single_round_rows(long groups_of_32, long groups_of_64, int compute_units) {
  return groups_of_32 <= compute_units ? 32 : groups_of_64 <= compute_units ? 64 : 128;
}

SkinnyPlan plan_skinny(int m, int n, int k, int compute_units) {
  const int chunks = (k + onebit::kChunkK - 1) / onebit::kChunkK;
  const int forced_rows = g_skinny_rows, forced_splits = g_split_k;
  // up to sixteen columns: single_round_rows
  // beyond: the largest row group that still gives about two workgroups per three compute units (measured: larger groups
  // re-read B less often, but idle compute units cost more)
  // (n > 32: two column fragments per row block, at most two row blocks per wavefront)
  const int enough = std::max(1, 160 * compute_units / 256);
  const int rows = forced_rows > 0 ? forced_rows
                   : n <= 16       ? single_round_rows((m + 31) / 32, (m + 63) / 64, compute_units)
                   : (m / 128 >= enough && n <= 32) ? 128 : (m / 64 >= enough) ? 64 : 32;
  if (forced_splits >= 1) return SkinnyPlan{rows, forced_splits > chunks ? chunks : forced_splits};
  const double image_row_bytes = n <= 16 ? 32.0 : n <= 32 ? 64.0 : 128.0;
  const double threshold = 400e3 * std::max(1.0, m / 4096.0);
  if (chunks < 32 || k * image_row_bytes < threshold) return SkinnyPlan{rows, 1};
  auto splits_for = [&](int r) {
    const int groups = (m + r - 1) / r;
    return std::min(compute_units / groups, chunks / 8);  // one workgroup per compute unit, eight chunks per workgroup
  };
  if (forced_rows > 0) {
    const int s = splits_for(rows);
    return SkinnyPlan{rows, s >= 2 ? s : 1};
  }
  if (const int s = splits_for(64); s >= 2) return SkinnyPlan{64, s};
  if (n <= 32)
    if (const int s = splits_for(128); s >= 2) return SkinnyPlan{128, s};
  return SkinnyPlan{rows, 1};
}

// Row group, tokens per workgroup and K splits over workgroups of wide_kernel: the plan with the least modelled time.
// A workgroup's wavefronts each multiply one K chunk per round; a round's time depends on the row group and the number of
// sixteen-token column tiles and grows with the share of compute units that load at the same time. Workgroups beyond one per
// compute unit pay the rounds again, less where two fit a compute unit (up to two column tiles on up to 64 rows). A split
// pays a second launch and the partial sums.
// Fitted to m = 1024 ... 28672, k = 1024 ... 22176, 17 ... 1024 tokens inside HIP graphs, when the kernel was slower than it is: it
// takes 0.78 to 0.96 of the modelled time now (median by class of plan). us of the chosen plan | of all tokens, or
// 64, per workgroup on 32 rows, unsplit: 28672 x 8192 x 48 22.3 (128 rows) | 40.4; 4096 x 11008 x 32 8.6 (32 rows, 16 tokens) | 12.0;
// 1024 x 4096 x 256 4.6 (64 rows, 16 tokens) | 6.6; 4096 x 4096 x 128 5.6 (64 rows, 32 tokens) | 7.4.
// total_groups: row groups of all products of the launch, for each of kWideRows.
const int kWideRows[3] = {32, 64, 128};
struct WidePlan {
  int rows, splits, tokens;
  double us;
};
WidePlan plan_wide(const long (&total_groups)[3], double results, int n, int k, bool plain, int least_splits,
                   int most_splits, int compute_units) {
  // [row group][column tiles - 1]
  static const double kBase[3][4] = {{2.75, 2.9, 2.9, 3.0}, {3.1, 3.3, 3.4, 3.6}, {3.7, 4.3, 5.8, 6.4}};
  static const double kRound[3][4] = {{0.74, 0.93, 1.48, 1.89}, {1.01, 1.26, 1.74, 2.24}, {1.88, 2.4, 2.75, 3.25}};
  static const double kLoad[3][4] = {{0.55, 0.55, 0.55, 0.55}, {0.23, 0.44, 0.5, 0.5}, {0.14, 0.24, 0.4, 0.4}};
  static const double kAgain[3][4] = {{0.57, 1.1, 1.0, 1.0}, {0.73, 0.9, 1.0, 1.0}, {1.0, 1.0, 1.0, 1.0}};
  static const double kSplitLines[3] = {1.17, 1.17, 1.05};  // k % 64 != 0: every second token's pieces straddle two lines
  // plain form, several column groups: a group's piece of a row of B is a part of a line, 32 to 128 bytes (4096 x 64 x 4096 in
  // four groups 11.0 us against 5.8 token-major, in two 7.1 against 5.1)
  static const double kColumns[4] = {2.3, 1.45, 1.4, 1.1};
  // and beyond 64 columns, with rows of B that begin inside a line, every round from the third on costs more (512 x 160 x 10112
  // in five rounds of 32-row groups 15.3 us, with K in three 11.0; up to 64 columns, where B is small, not: 1280 x 56 x 7520 in
  // two groups 10.4, in one 12.9)
  static const double kFurther[3] = {0.18, 0.06, 0.0};
  const bool cut_lines = n > onebit::kSkinnyMaxN && n % 64;
  // The row groups that multiply one token group run on different XCDs, and each XCD fetches its own copy of x: with more x
  // than fits an XCD's L2 (4 MB) that is what a launch of few rows waits for (fitted to us measured | modelled without it: 896 x 24256
  // x 704 45 | 29, 1088 x 13888 x 1758 62 | 38, 640 x 17536 x 676 30 | 19. In strips these take 42, 59 and 23 as products, the main
  // kernel 34, 46 and 26, and 29, 59 and 21 as layers, the main kernel 35, 42 and 26).
  constexpr double kFetchBytesPerUs = 5.6e6;
  const double xcds = std::max(1, compute_units / 32);
  const int chunks = (k + onebit::kChunkK - 1) / onebit::kChunkK;
  WidePlan best{g_skinny_rows > 0 ? g_skinny_rows : 32, 1, std::min(n, onebit::kSkinnyMaxN), 1e30};
  for (int width = 1; width <= 4; ++width) {
    const int groups = (n + 16 * width - 1) / (16 * width);
    const int tokens = ((n + groups - 1) / groups + 7) / 8 * 8, tiles = (tokens + 15) / 16;
    if (tiles != width) continue;  // the same groups as with narrower ones
    for (int r = 0; r < 3; ++r) {
      if (g_skinny_rows > 0 && g_skinny_rows != kWideRows[r]) continue;
      for (int s : {1, 2, 3, 4, 6, 8}) {
        if (g_split_k >= 1) s = g_split_k;
        s = std::min(std::min(s, most_splits), chunks);
        if (s < least_splits) continue;
        const int rounds = ((chunks + s - 1) / s + 7) / 8;
        const double load = (double)total_groups[r] * groups * s / compute_units;
        const double work = rounds * kRound[r][tiles - 1] * (1.0 + kLoad[r][tiles - 1] * std::min(1.0, load)) *
                            (!plain       ? (k % 64 ? kSplitLines[r] : 1.0)
                             : groups > 1 ? kColumns[tiles - 1] * (cut_lines ? 1.0 + kFurther[r] * std::max(0, rounds - 2) : 1.0)
                                          : 1.0);
        double us = kBase[r][tiles - 1] + work;
        if (load > 1.0)
          us += (std::ceil(load) - 1.0) * (work * kAgain[r][tiles - 1] + (kBase[r][tiles - 1] - 1.5) * (r < 2 ? 0.4 : 1.0));
        us = std::max(us, 3.0 + std::min((double)total_groups[r], xcds) * n * k * 2.0 / kFetchBytesPerUs);
        if (s > 1) us += 2.6 + 0.15 * s + (s + 1) * 4.0 * results / 5.0e6;
        if (us < best.us) best = WidePlan{kWideRows[r], s, tokens, us};
        if (g_split_k >= 1 || s == most_splits) break;
      }
    }
  }
  return best;
}

// Whether wide_kernel walks its grid in strips of two column groups. Dealt over the XCDs by row groups, every XCD fetches all of x
// and, where their number is no multiple of eight, the same rows of the weight for several of the column groups; in strips it fetches
// a few column groups of x and a part of the rows. That pays where all of x does not fit an XCD's L2 (4 MB), and where x and the
// weight are large enough for the second fetch to show, the earlier the more XCDs repeat it. us inside HIP graphs, weights from HBM, dealt
// | strips: x of 4 MB and more: 2048 x 256 x 8192 14.1 | 12.3, layers 1024 x 4096 with 1000 tokens 14.5 | 12.6, 6784 x 9984 with
// 537 54.8 | 52.2; an odd number of row groups: layers 960 x 6528 with 415 10.5 | 8.0, 3456 x 4640 with 135 10.1 | 9.2, 1984 x 2784 with
// 123 5.3 | 4.8; below: layers 512 x 1024 with 500 3.15 | 3.40, 4096 x 4096 with 200 8.0 | 8.7, products 4096 x 256 x 4096 9.4 |
// 10.1, 1024 x 64 x 4096 5.0 | 5.35, 704 x 48 x 2976 4.75 | 4.55. On 700 calls in several column groups this rule is 3.8 % faster in
// the mean than strips wherever there are several (with their parameters loaded); eight are more than 2 % slower.
bool wide_in_strips(int m, int n, int k, const WidePlan& plan, bool plain, int compute_units) {
  const int column_groups = (n + plan.tokens - 1) / plan.tokens, row_groups = (m + plan.rows - 1) / plan.rows;
  // a layer's x of up to 64 tokens lies in every L2; the walk is made for eight XCDs of 32 compute units
  if (column_groups < 2 || (!plain && n <= onebit::kSkinnyMaxN) || compute_units != 256) return false;
  const double x = 2.0 * n * k, both = x + 0.1875 * m * k;
  return x >= 4e6 || (row_groups % 2 ? both >= 1.5e6 : row_groups % 4 ? both >= 3.5e6 : false);
}

LaunchPlan choose_launch(int m, int n, int k, bool b_16_byte_aligned, int compute_units) {
  LaunchPlan plan{};
  // 32 < n <= 64: every 64-row workgroup of the split-K kernel stages all of B, which the main kernel's tiles overtake
  // from about 48k rows on (n = 64: 28672 x 8192 32 us against 42; 32768 x 4096 20 against 26; 49152 x 4096 32.5
  // against 34.4; 65536 x 8192 66 against 68, at n = 40 77 against 66; 131072 x 2048 51 against 35)
  const bool skinny_shape = n <= 32 || (n <= onebit::kSkinnyMaxN && m <= 40960);
  if (skinny_shape && g_skinny_enabled) {
    const SkinnyPlan sk = plan_skinny(m, n, k, compute_units);
    plan.split_k_kernel = 1;
    plan.rows_or_tile = sk.rows;
    plan.splits = sk.splits;
    return plan;
  }
  const GemmPlan gemm = plan_gemm(m, n, k, compute_units);
  plan.rows_or_tile = gemm.tile;
  plan.splits = gemm.splits;
  plan.model_us = gemm.us;
  // B rows that are not 16-byte aligned: pad a copy (one extra pass over B) unless the problem is too small for that
  // to pay against the element-copy variant of the kernel
  const bool b_in_place = n % 8 == 0 && b_16_byte_aligned;
  plan.pad_b = !b_in_place && (size_t)k * n >= 65536 && g_pad_b;
  return plan;
}

// wide_kernel against the main kernel. Both models err, and by how much depends on the plans. A line of 0.81 to 0.88 was drawn where
// about as few calls were slower on either side, on an earlier wide_kernel, whose model has it too slow now wherever its workgroups
// have a compute unit each (in several rounds it is right: 64-row groups of 4992 x 1024 with 270 tokens, 468 of them, 8.7 us, 6.7 on
// the main kernel at 1.17 of its modelled time). There the line is 1.05; main kernel | wide_kernel, us inside HIP graphs, weights from
// HBM, random calls that it moves: 22 layers of one whole tile per K range 0.70 to 0.98 of the time, median 0.84 (3520 x 1248 with 206
// tokens 8.6 | 6.0, 2624 x 7584 with 630 33.9 | 24.0), 44 products 0.51 to 1.03, median 0.79 (1088 x 672 with 416 columns 6.9 | 4.3, 3840 x
// 7136 with 512 29.0 | 23.0, 1856 x 2400 with 471 17.4 | 10.9), 135 layers where the main kernel splits K 0.54 to 1.08, median 0.86 (704 x
// 7456 with 985 19.3 | 13.5). A long K is where both models' errors grow: 38 more such layers, from 60 chunks on in groups of 64 tokens
// against the 256 x 128 tile and from 71 on in groups of 32 and 64 rows, are 0.91 to 1.14 of the time, mean 1.00 (2048 x 27552 with 846
// 61.6 | 70.2, 3776 x 26336 with 496 61.9 | 67.0, 1280 x 22304 with 295 24.4 | 26.4; 1344 x 24448 with 345 25.9 | 24.0), and stay, on 64
// rows but for what is below 0.9 of the modelled time (0.86 to 0.94 but for two of 1.01 and 1.07). Not moved: products where the main
// kernel splits K (768 x 8192 with 616 16.3 | 17.4) or has the 256 x 128 tile (5440 x 13120 with 168 30.9 | 34.4); and layers in groups
// of other than 32 or 64 tokens where it splits K, products with a workgroup for every compute unit or 32-row groups. Those lines are not
// where the measurements end: some calls beyond would gain (4096 x 4096 with 512 20.3 | 16.9, 512^3 4.8 | 3.6; 1024^3 6.5 | 6.5), others
// not (layers of 1344 x 9216 with 969 and of 640 x 17536 with 676), and they have not been timed over the ranges.
// The sums are fp32 on both sides and in another order. Their relative error against 64 bits, main kernel | wide_kernel, 1e-8: layers that
// it splits 704 x 7456 with 985 6.0 | 6.7, 960 x 17696 with 329 7.4 | 8.0, 3328 x 17440 with 465 8.9 | 8.0, 576 x 10848 with 484 7.3 |
// 6.5; others 5.8 | 5.6 (1216 x 3808 with 1077); products 4.8 | 4.7, 7.7 | 6.9, 2.8 | 2.5.
// Where wide_kernel splits K the line is 0.96 for layers (0.78 to 1.03, median 0.88) and, with three splits or more, for products (0.73
// to 1.03, median 0.87; in two splits 0.95 to 1.13, in few rows on 64-row groups up to 1.05).
// Up to 64 columns the main kernel is the other plan beyond 40960 rows only, where a wavefront of wide_kernel has one short round
// of work per workgroup and the workgroups come in many rounds, outside what its model was fitted to: the line is the length of
// K, from which on wide_kernel is faster at 45056 to 262144 rows (us, wide | main, 48 and 64 tokens: 65536 x 1024 15.8 | 15.6 and
// 16.2 | 16.9, x 4096 28.4 | 33.2 and 32.5 | 33.5, x 8192 44.7 | 61.5 and 51.5 | 62.8; 45056 x 3616 24.6 | 26.5 and 27.1 | 26.7,
// x 4096 23.9 | 27.3 and 28.5 | 27.5). With k % 64 != 0, where every second token's pieces straddle two lines, it lies twice as far out
// (45056 x 4128 with 48 tokens 30.3 | 28.7, x 8224 45.7 | 51.4). Where the main kernel would split K,
// wide_kernel in any case (41024 x 7936 and x 8160, 56 and 64 tokens: 44.1 to 47.8 against 55.5 to 59.4).
bool wide_is_faster(const WidePlan& wide, const LaunchPlan& launch, int m, int n, int k, bool plain, int compute_units) {
  const int chunks = (k + onebit::kChunkK - 1) / onebit::kChunkK;
  if (n <= onebit::kSkinnyMaxN) return launch.splits > 1 || chunks >= (n <= 48 ? 16 : 32) * (k % 64 ? 2 : 1);
  const long workgroups = (long)((m + wide.rows - 1) / wide.rows) * ((n + wide.tokens - 1) / wide.tokens);
  const bool many_splits = !plain || (wide.splits >= 3 && (wide.rows == 128 || m >= 1024));
  double line = wide.splits > 1                                 ? (many_splits ? 0.96 : 0.92)
                : launch.rows_or_tile == onebit::kTile256x128w8 ? 0.81
                : plain                                         ? 0.85
                : launch.splits > 1                             ? 0.87
                                                                : 0.88;
  if (wide.splits == 1 && workgroups <= compute_units) {
    if (plain) {
      if (launch.rows_or_tile != onebit::kTile256x128w8 && launch.splits <= 1 && wide.rows >= 64 && workgroups < compute_units) line = 1.05;
    } else if (launch.splits <= 1) {
      line = 1.05;
    } else if (wide.tokens == 32 || wide.tokens == 64) {
      const bool main_256x128 = launch.rows_or_tile == onebit::kTile256x128w8;
      const bool long_k = wide.tokens == 64 ? main_256x128 && chunks >= 60 : wide.rows == 64 && chunks > 70;
      if (!long_k) line = 1.05;
      else if (!main_256x128) line = 0.9;
    }
  }
  return wide.us < line * launch.model_us;
}

// Least K splits of wide_kernel in the place of a `launch` that splits K, up to 64 columns: its model, fitted to weights that lie
// in the Infinity Cache, has the unsplit plan ahead too often when they come from HBM.
// Plain form (us with weights from HBM, that kernel's split plan | wide_kernel unsplit | in two): 4096 x 11008 with 24 columns
// 10.9 | 11.2 | 10.6, 2048 x 9600 with 24 and 32 10.2 | 10.5 | 9.6 and 9.6 | 11.3 | 9.2, 4096 x 9600 with 64 14.0 | 14.9 | 13.1,
// 2048 x 8192 with 32 9.0 | 9.5 | 8.3; unsplit allowed at 8192 x 8192 with 64 16.5 | 14.3 | 15.4, 4096 x 8192 with 24 9.9 | 9.1 | 9.1.
// Token-major form, whose images cost less: split where that kernel splits over 128-row groups (10241 to 16384 rows) and the
// workgroups' copies of x are long (11008 x 28672 with 24 and 32 tokens 27.6 | 30.1 | 27.4 and 30.3 | 34.7 | 29.5, not 11008 x
// 20480 with 17 20.7 | 19.7 | 21.4), and where it splits a very long K three times or more (5120 x 13824 with 17 tokens
// 11.4 | 12.2 | 11.7, in three 10.8).
int wide_least_splits(const LaunchPlan& launch, int n, int k, bool plain) {
  if (launch.splits <= 1 || n > onebit::kSkinnyMaxN) return 1;
  const int chunks = (k + onebit::kChunkK - 1) / onebit::kChunkK;
  if (plain) return chunks > 32 || (n > 24 && n <= 32) ? 2 : 1;
  if (!launch.split_k_kernel) return 1;
  if (launch.rows_or_tile == 128) return (long)k * n >= 480000 ? 2 : 1;
  return n <= 32 && launch.splits >= 3 && chunks >= 50 ? 2 : 1;
}

// The linear layer's plan: wide = wide_kernel with `wide_plan`, else `launch` as for a product with an aligned B.
// Up to sixteen tokens the split-K kernel; beyond, wide_kernel in that kernel's place and where it is faster than the main
// kernel. A layer call splits K into no more parts than the other kernel's plan would and uses the same buffer, so a call needs
// no more memory than it would there, and what can be captured without a warm-up stays so.
struct LinearPlan {
  bool wide;
  WidePlan wide_plan;
  LaunchPlan launch;
};
LinearPlan plan_linear(int m, int tokens, int k, int compute_units) {
  LinearPlan plan{};
  plan.launch = choose_launch(m, tokens, k, true, compute_units);
  if (tokens <= onebit::kSkinnyTokens || !g_skinny_enabled) return plan;
  const long groups[3] = {(m + 31) / 32, (m + 63) / 64, (m + 127) / 128};
  if (!plan.launch.split_k_kernel && g_tile_config >= 0) return plan;
  if (tokens > onebit::kSkinnyMaxN && groups[2] * ((tokens + 63) / 64) > 2L * compute_units) return plan;
  plan.wide_plan = plan_wide(groups, (double)m * tokens, tokens, k, false, wide_least_splits(plan.launch, tokens, k, false),
                             plan.launch.splits, compute_units);
  plan.wide = plan.launch.split_k_kernel || wide_is_faster(plan.wide_plan, plan.launch, m, tokens, k, false, compute_units);
  return plan;
}

// The product's: wide_kernel in the place of `launch` for 17 columns or more where that reads B in place or through its padded
// copy: in the place of the split-K kernel, but for some of 32 columns, and where it is faster than the main kernel. It splits K
// into no more parts than `launch` and uses the same buffers, so a call needs no memory that it would not need there, and what
// can be captured without a warm-up stays so. It may split into fewer or not at all: a split pays a second launch and fp32 sums
// through memory (us, split in two -> unsplit: 1024 x 128 x 2048 6.1 -> 3.8, 4096 x 96 x 4096 10.8 -> 7.2, 5120 x 128 x 8192
// 20.0 -> 13.3).
WidePlan plan_wide_product(const LaunchPlan& launch, int m, int n, int k, bool b_readable, int compute_units) {
  WidePlan none{0, 1, 0, 0.0};
  const long groups[3] = {(m + 31) / 32, (m + 63) / 64, (m + 127) / 128};
  // 32 columns, whole rows of an image: skinny_kernel is as fast or faster in one round of 128-row groups, in its split plans
  // from 3073 rows on, and where K is so short that its chunks do not fill a round of the sixteen wavefronts of its 32-row
  // groups, one per compute unit (us, skinny_kernel | wide_kernel: 20480 x 4096 10.4 | 11.2, 28672 x 5536 14.2 | 15.0, 11008 x
  // 20480 22.9 | 23.5; 4096 x 11008 10.5 | 11.1, 5120 x 8192 10.2 | 10.7, 2048 x 9600 9.5 | 8.3; 2048 x 1056 3.71 | 3.85, but in
  // two rounds of workgroups 9920 x 992 5.6 | 4.1, 8512 x 1088 6.3 | 4.8; 4096 x 4096 5.55 | 5.17, 40960 x 4096 19.7 | 16.6)
  const bool one_short_round = launch.rows_or_tile == 32 && k <= 5 * onebit::kChunkK && groups[0] <= compute_units;
  if (n == 32 && g_skinny_rows <= 0 && launch.split_k_kernel && groups[2] <= compute_units &&
      (launch.rows_or_tile == 128 || (launch.splits > 1 ? groups[0] * 8 > 3L * compute_units : one_short_round)))
    return none;
  if (n <= 16 || !g_skinny_enabled || g_tile_config >= 0 || groups[2] * ((n + 63) / 64) > 2L * compute_units) return none;
  if (!b_readable) return none;
  const WidePlan plan = plan_wide(groups, (double)m * n, n, k, true, wide_least_splits(launch, n, k, true), launch.splits,
                                  compute_units);
  if (plan.us == 1e30 || (!launch.split_k_kernel && !wide_is_faster(plan, launch, m, n, k, true, compute_units))) return none;
  return plan;
}

// Whether a ragged B (n % 8 != 0, 16-byte aligned) is read where it lies instead of through a padded copy. The copy costs a launch
// and a pass, 4 to 5 us and 4 bytes per value at 5.5 TB/s; rows that start at an odd value cost the asynchronous copies 2.4 times the
// load path (read_as_ragged), which the smaller tiles are short of.
// Even n: always but on few rows and a short K up to 32 columns, where skinny_kernel has as little to read: 10 calls 0.94 to 1.03 of
// its time, with a C 16 of 0.96 to 1.09 (1600 x 320 with 22 3.8 | 4.2; 9600 x 320 with 28 6.7 | 4.7). us inside HIP graphs, padded
// copy, or skinny_kernel up to 64 columns | in place: 4096 x 4096 with 34 / 100 / 500 / 2050 columns 9.0 | 6.4, 12.2 | 9.7, 25.9 | 21.5,
// 53.3 | 46.1, 28672 x 8192 with 50 39.8 | 25.4, 11008 x 4096 with 1002 57.9 | 54.2, 704 x 1760 with 8142 28.5 | 19.5.
// Odd n on the main kernel, by tile: 512 x 128 and one 256 x 128 or eight-wavefront 128 x 128 per compute unit, where a stage takes long
// enough: 37 of 37 calls faster, 11008 x 4096 with 1001 56.8 | 52.1, 896 x 6144 with 5995 72.8 | 46.8. 256 x 128, two per compute unit: up
// to one and a half rounds (in four 11776 x 6624 with 6257 460 | 478) of up to 15 chunks (109 calls 0.86 to 1.04 of the time, mean 0.95,
// 4992 x 928 with 3589 37.0 | 33.9; of 41 longer ones 0.93 to 1.09, mean 1.01, 21312 x 3872 with 969 96.4 | 100.3). 64 x 128, and 128 x 128
// in two K groups: on a short K, shorter where a copy of few columns is soon made (218 calls 0.68 to 1.00, mean 0.84, 1600 x 896 with 1243
// 13.4 | 11.7; 13760 x 1888 with 65 13.7 | 16.1, 26112 x 1536 with 85 14.1 | 14.9) and, but for the first, few rows (212 calls 0.63 to
// 1.07, median 0.83, 704 x 9728 with 2889 62.9 | 58.1; six are more than 3 % slower, where the copy's row length suits the caches: 640 x
// 7008 with 1977 34.6 | 36.9, with 2197 43.4 | 37.2; 4672 x 8064 with 539 40.5 | 45.2).
// Odd n on wide_kernel: up to 64 columns, where skinny_kernel is the other one (4096 x 4096 with 49 15.0 | 7.5, 28672 x 8192 with 33 47 |
// 28), but not where that splits K and 32-row groups of 24, 40 or 48 columns do not (K of 32 chunks, 4160 x 8192 with 35 14.3 | 18.7,
// 2368 x 8192 with 17 9.4 | 11.5, all of 46 calls 1.04 to 1.31 of the time); in groups of 16, 32 or 64 of more columns (512 x 1856 with 555
// 10.4 | 6.8; in groups of 48 7360 x 4192 with 87 14.7 | 17.0). It would be faster on fewer rows and a longer K too (896 x 1696 with 39
// 6.7 | 4.4, 2048 x 4832 with 233 14.9 | 11.9): these two lines, by m and chunks, are not where the measurements end, the calls beyond
// them have not been timed over the ranges.
bool ragged_in_place(int m, int n, int k, const LaunchPlan& launch, const WidePlan& wide, int compute_units) {
  const int chunks = (k + onebit::kChunkK - 1) / onebit::kChunkK;
  if (n % 2 == 0) return !launch.split_k_kernel || n > 32 || m > 8192 || chunks > 4;
  if (wide.rows) {
    if (launch.splits > 1 && wide.splits == 1 && wide.rows == 32 && wide.tokens % 32 != 0) return false;
    if (n <= onebit::kSkinnyMaxN) return m > 2048 || (m > 1088 && chunks <= 16);
    return (wide.tokens == 16 || wide.tokens == 32 || wide.tokens == 64) && chunks <= 16;
  }
  const bool short_k = chunks <= (n <= 224 ? 5 : 7);
  switch (launch.rows_or_tile) {
    case onebit::kTile512x128w8: case onebit::kTile512x128m16: case onebit::kTile256x128w8: case onebit::kTile128x128w8: return true;
    case onebit::kTile256x128w: return chunks <= 15 && (long)((m + 255) / 256) * ((n + 127) / 128) <= 3L * compute_units;
    case onebit::kTile64x128: return short_k;
    case onebit::kTile128x128k2: case onebit::kTile64x128k2: return short_k || m <= 1024;
    default: return false;
  }
}

// Everything decided about a product: wide.rows != 0: wide_kernel, else `launch`; pad_b: B is read through a padded copy. A ragged B
// keeps it where the call splits K beyond 64 columns: their tests pin its place in the workspace beside the partial sums.
// small_pad: a padded copy that the plan does not count on can be had.
struct ProductPlan {
  LaunchPlan launch;
  WidePlan wide;
  bool pad_b;
};
template <class SmallPad>
ProductPlan plan_product(int m, int n, int k, bool b_16_byte_aligned, int compute_units, SmallPad&& small_pad) {
  ProductPlan plan{};
  plan.launch = choose_launch(m, n, k, b_16_byte_aligned, compute_units);
  const LaunchPlan& launch = plan.launch;
  const bool b_in_place = n % 8 == 0 && b_16_byte_aligned;
  // (a forced tile without a build for it reads the padded copy: 4096 x 1002 x 4096 in element copies more than ten times as long)
  const bool ragged = n % 8 != 0 && n >= 8 && b_16_byte_aligned && (launch.split_k_kernel || onebit::tile_reads_ragged(launch.rows_or_tile));
  plan.pad_b = launch.pad_b || (!launch.split_k_kernel && !b_in_place && !ragged && g_pad_b && small_pad());
  plan.wide = plan_wide_product(launch, m, n, k, b_in_place || plan.pad_b || ragged, compute_units);
  if (ragged) {
    const bool in_place = ragged_in_place(m, n, k, launch, plan.wide, compute_units);
    if (launch.split_k_kernel && !in_place) plan.wide = WidePlan{0, 1, 0, 0.0};  // skinny_kernel
    if (in_place && (plan.wide.rows ? plan.wide.splits : launch.splits) <= 1) plan.pad_b = false;
  }
  return plan;
}

// Workspace of one call that the caller cannot let allocate: `base` is this device's copy of the file-scope array
// g_static_scratch (see onebit_sparse_matmul_prepared_static), `bytes` its size.
struct FixedScratch {
  unsigned char* base;
  size_t bytes;
};

// Splits that a plan's `splits` come to: none of them empty.
int full_splits(int chunks, int splits) {
  const int per_split = (chunks + splits - 1) / splits;
  return (chunks + per_split - 1) / per_split;
}

using DeviceLock = std::unique_lock<std::recursive_mutex>;

// K split of a split-K kernel launch: the split geometry and the partial-sum buffer (the caller's fixed workspace, or
// the library-owned buffer of this device and stream). With the latter `lock` holds the device's lock on return and the caller
// keeps it until both kernels are enqueued: another thread's call on the stream must not come between them, and must not
// replace the buffer before they are enqueued.
// most_splits: of the plan that wide_kernel's replaces, at least `splits`. The buffer is made large enough for that many: how
// far wide_kernel splits changes from one column count to the next in both directions, so a call of fewer columns would
// otherwise replace a buffer that a graph captured with more of them still reads.
int setup_skinny_split(onebit::SkinnyArgs& args, int splits, int most_splits, hipStream_t stream, const FixedScratch* fixed,
                       DeviceLock& lock) {
  args.splits = 1;
  if (splits <= 1) return ONEBIT_OK;
  args.chunks_per_split = (args.kc_total + splits - 1) / splits;
  args.splits = full_splits(args.kc_total, splits);
  if (args.splits <= 1) return ONEBIT_OK;
  const size_t split_bytes = (size_t)args.m * args.n * sizeof(float), bytes = args.splits * split_bytes;
  if (fixed) {
    if (bytes > fixed->bytes)
      return fail(ONEBIT_ERR_ARGUMENT,
                  "this shape needs %zu bytes of scratch (%d K splits of %d x %d fp32 partial sums); the static "
                  "workspace of the non-allocating entry point holds %zu", bytes, args.splits, args.m, args.n, fixed->bytes);
    args.split_ws = reinterpret_cast<float*>(fixed->base);
    return ONEBIT_OK;
  }
  int device = 0;
  ONEBIT_HIP(hipGetDevice(&device));
  if (device < 0 || device >= kMaxDevices) return fail(ONEBIT_ERR_ARGUMENT, "device ordinal %d not supported", device);
  DeviceState& st = g_dev[device];
  lock = DeviceLock(st.mu);
  Buffer& ws = st.split_ws[stream];
  if (int rc = grow(&ws.ptr, &ws.bytes, bytes, stream, full_splits(args.kc_total, most_splits) * split_bytes); rc != ONEBIT_OK)
    return rc;
  args.split_ws = static_cast<float*>(ws.ptr);
  return ONEBIT_OK;
}

// Least size of a padded-copy buffer: that of any B below the 65536 values from which the plan pads (rows of one column grow
// eightfold). Growing frees the old buffer, which a graph captured earlier still reads; a small B never makes one grow.
constexpr size_t kLeastPadBytes = size_t(65536) * 8 * sizeof(_Float16);

// Whether a padded copy of a small B (the plan does not count on one) can be made without failing a call that went through
// without it: never inside a capture that would have to allocate, and never in a fixed workspace, whose size the plan is
// checked against.
bool small_pad_available(size_t bytes, hipStream_t stream, const FixedScratch* fixed) {
  int device = 0;
  if (fixed || hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return false;
  DeviceState& st = g_dev[device];
  std::lock_guard<std::recursive_mutex> lock(st.mu);
  Buffer& pb = st.b_pad[stream];
  if (bytes <= pb.bytes) return true;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone &&
      grow(&pb.ptr, &pb.bytes, std::max(bytes, kLeastPadBytes), stream) == ONEBIT_OK)
    return true;
  // the call goes on without the copy: nothing of the attempt may show in it
  (void)hipGetLastError();
  g_last_error.clear();
  return false;
}

int matmul_prepared_impl(const void* prepared, const void* b, const void* c, void* d, int m, int n, int k, float alpha,
                         float beta, int c_dtype, int d_dtype, hipStream_t stream, const FixedScratch* fixed = nullptr) {
  if (!prepared || !b || !d) return fail(ONEBIT_ERR_ARGUMENT, "null operand pointer");
  if (beta != 0.f && !c) return fail(ONEBIT_ERR_ARGUMENT, "c must not be null when beta != 0");
  const int kc_total = (k + onebit::kChunkK - 1) / onebit::kChunkK;

  const int compute_units = current_compute_units();
  const bool b_aligned = (reinterpret_cast<uintptr_t>(b) & 15) == 0;
  // A small B that the main kernel cannot read in place is described as read by element copies; a padded copy is many times
  // faster (1152 x 77 x 640 61 -> 6 us) and is made wherever its buffer is there or can be had.
  const size_t pad_bytes = (size_t)k * ((size_t)(n + 7) / 8 * 8) * sizeof(_Float16);
  const ProductPlan product =
      plan_product(m, n, k, b_aligned, compute_units, [&] { return small_pad_available(pad_bytes, stream, fixed); });
  const LaunchPlan& plan = product.launch;
  const WidePlan& wide = product.wide;
  const bool pad_b = product.pad_b;
  if (plan.split_k_kernel) {
    onebit::SkinnyArgs args{};
    args.prep = static_cast<const uint8_t*>(prepared);
    args.b = static_cast<const _Float16*>(b);
    args.c = c;
    args.d = d;
    args.m = m; args.n = n; args.k = k;
    args.kc_total = kc_total;
    args.alpha = alpha; args.beta = beta;
    args.c_f16 = c_dtype == ONEBIT_DTYPE_F16;
    args.d_f16 = d_dtype == ONEBIT_DTYPE_F16;
    args.tokens_per_group = wide.tokens;
    args.strips = wide.rows && wide_in_strips(m, n, k, wide, true, compute_units);
    args.ldb = n;
    DeviceLock lock;
    if (int rc = setup_skinny_split(args, wide.rows ? wide.splits : plan.splits, plan.splits, stream, fixed, lock); rc != ONEBIT_OK)
      return rc;
    ONEBIT_HIP(wide.rows ? onebit::launch_wide(args, wide.rows, stream) : onebit::launch_skinny(args, plan.rows_or_tile, stream));
    return ONEBIT_OK;
  }

  if (onebit::prepared_bytes(m, k) >= (size_t(1) << 32))
    return fail(ONEBIT_ERR_ARGUMENT,
                "the main kernel addresses the prepared operand with 32-bit offsets: m x k = %d x %d needs %zu bytes, "
                "the limit is 4 GiB (about 22.9e9 weights); split the weight by rows", m, k, onebit::prepared_bytes(m, k));
  onebit::GemmArgs args{};
  args.prep = static_cast<const uint8_t*>(prepared);
  args.b = static_cast<const _Float16*>(b);
  args.c = c;
  args.d = d;
  args.m = m; args.n = n; args.k = k;
  args.kc_total = kc_total;
  args.alpha = alpha; args.beta = beta;
  args.c_f16 = c_dtype == ONEBIT_DTYPE_F16;
  args.d_f16 = d_dtype == ONEBIT_DTYPE_F16;
  const int tile = plan.rows_or_tile;
  const int splits = wide.rows ? wide.splits : plan.splits;
  auto launch = [&]() -> hipError_t {
    if (!wide.rows) return onebit::launch_gemm(args, tile, stream);
    onebit::SkinnyArgs w{};
    w.prep = args.prep;
    w.b = args.b;
    w.c = c;
    w.d = d;
    w.m = m; w.n = n; w.k = k;
    w.kc_total = kc_total;
    w.alpha = alpha; w.beta = beta;
    w.c_f16 = args.c_f16;
    w.d_f16 = args.d_f16;
    w.splits = args.splits;
    w.chunks_per_split = args.chunks_per_split;
    w.split_ws = args.split_ws;
    w.tokens_per_group = wide.tokens;
    w.strips = wide_in_strips(m, n, k, wide, true, compute_units);
    w.ldb = n;
    if (pad_b) {
      if (hipError_t st = onebit::launch_pad_b(args.b, args.b_pad, k, n, stream); st != hipSuccess) return st;
      w.b = args.b_pad;
      w.ldb = (n + 7) / 8 * 8;
    }
    return onebit::launch_wide(w, wide.rows, stream);
  };
  if (splits > 1 || pad_b) {
    size_t split_bytes = 0, most_bytes = 0;
    if (splits > 1) {
      args.chunks_per_split = (kc_total + splits - 1) / splits;
      args.splits = full_splits(kc_total, splits);
      split_bytes = (size_t)args.splits * m * n * sizeof(float);
      most_bytes = (size_t)full_splits(kc_total, plan.splits) * m * n * sizeof(float);  // see setup_skinny_split
    }
    if (fixed) {
      // partial sums first, the padded copy of B behind them on the next 256-byte boundary; both are written in
      // full by this call's own kernels before they are read, so nothing has to start at zero
      const size_t pad_at = (split_bytes + 255) & ~size_t(255), pad_need = pad_b ? pad_bytes : 0;
      if (pad_at + pad_need > fixed->bytes)
        return fail(ONEBIT_ERR_ARGUMENT,
                    "this shape needs %zu bytes of scratch (%d K splits of %d x %d fp32 partial sums, %zu bytes of "
                    "padded B); the static workspace of the non-allocating entry point holds %zu",
                    pad_at + pad_need, splits > 1 ? args.splits : 0, m, n, pad_need, fixed->bytes);
      if (splits > 1) args.split_ws = reinterpret_cast<float*>(fixed->base);
      if (pad_b) args.b_pad = reinterpret_cast<_Float16*>(fixed->base + pad_at);
      ONEBIT_HIP(launch());
      return ONEBIT_OK;
    }
    int device = 0;
    ONEBIT_HIP(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices) return fail(ONEBIT_ERR_ARGUMENT, "device ordinal %d not supported", device);
    DeviceState& st = g_dev[device];
    std::lock_guard<std::recursive_mutex> lock(st.mu);
    if (splits > 1) {
      Buffer& ws = st.split_ws[stream];
      if (int rc = grow(&ws.ptr, &ws.bytes, split_bytes, stream, most_bytes); rc != ONEBIT_OK) return rc;
      args.split_ws = static_cast<float*>(ws.ptr);
    }
    if (pad_b) {
      Buffer& pb = st.b_pad[stream];
      if (int rc = grow(&pb.ptr, &pb.bytes, std::max(pad_bytes, kLeastPadBytes), stream); rc != ONEBIT_OK) return rc;
      args.b_pad = static_cast<_Float16*>(pb.ptr);
    }
    ONEBIT_HIP(launch());
    return ONEBIT_OK;
  }
  ONEBIT_HIP(launch());
  return ONEBIT_OK;
}

// Whether fp32 activations of that many tokens go through the kernel that rounds them itself (skinny_kernel).
bool takes_f32(int tokens) { return tokens <= onebit::kSkinnyTokens && g_skinny_enabled; }

// Whether skinny_kernel on fp32 activations is faster than converting them and running it on fp16 ones. Every workgroup reads all of
// x of its K range, so fp32 costs a compute unit half of these bytes more, and beyond eight tokens an image comes in two batches, the
// second requested behind the first; both hide behind the weights until they are many. The conversion costs about 2 us whatever the
// size, and the host 4 us, which a call outside a graph hides behind its kernel only if that takes 9 us. us inside HIP graphs, weights
// from HBM, converted | read as fp32: 4096 x 8192 with 16 tokens 8.5 | 7.9, x 11008 with 9 / 12 / 16 8.6 | 7.4, 9.1 | 8.3, 9.2 | 9.7;
// 8192 x 14336 with 8 / 9 10.0 | 9.0, 10.3 | 9.4; 7168 x 20480 with 8 / 16 11.0 | 11.0, 16.7 | 19.7; 11008 x 28672 with 5 / 16 20.1 |
// 19.1, 26.1 | 32.7; two rounds of workgroups: 49152 x 2048 with 16 13.7 | 13.8, x 4096 18.1 | 19.4. Of 170 calls near the lines one that
// is read is more than 5 % slower than converted (832 x 9088 with 16, 8.2 | 8.7). The lines were drawn when nine to fifteen tokens took
// the loads of sixteen in branches: 20 calls that are converted would be 5 to 22 % faster read, most of nine to thirteen tokens (4608 x
// 12448 with 10 10.2 | 8.3). Call after call without a graph: 4096 x 9600 with 16 10.1 | 8.9, x 11008 with 13 / 16 10.2 | 8.6, 10.2 |
// 9.5, 5120 x 13824 with 12 10.2 | 9.8, 8192 x 14336 with 9 10.2 | 9.2, 11008 x 28672 with 16 26.9 | 34.0.
bool reading_f32_is_faster(int tokens, int m, int k, int compute_units, hipStream_t stream) {
  // read whatever the plan: no row group is smaller than 32, a split reads less (spares a small call the second plan)
  const long most_rounds = (m / 32 + compute_units - 1) / compute_units;
  if ((double)k * most_rounds * (tokens + 16) < 150e3) return true;
  const LaunchPlan plan = plan_linear(m, tokens, k, compute_units).launch;
  const int splits = full_splits((k + onebit::kChunkK - 1) / onebit::kChunkK, plan.splits);
  const long workgroups = (long)((m + plan.rows_or_tile - 1) / plan.rows_or_tile) * splits;
  const long rounds = (workgroups + compute_units - 1) / compute_units;
  const double values = (double)k / splits * rounds;  // of a token that a compute unit reads
  if (tokens <= 8) return values * tokens < 150e3;
  const double work = values * (tokens + 16);
  if (rounds > 1 || work < 307e3 || work >= 390e3) return work < (rounds > 1 ? 150e3 : 307e3);
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capture) == hipSuccess) return capture == hipStreamCaptureStatusNone;
  (void)hipGetLastError();  // the default stream, another one being captured: the launch is not to report this
  return false;
}

// The layer's product on 16-bit activations of either type, or up to sixteen tokens of fp32 ones (x_dtype).
int linear_prepared_impl(const void* prepared, const void* x, const void* bias, void* y, int tokens, int m, int k, int x_dtype,
                         int bias_dtype, int y_dtype, hipStream_t s) {
  if (!prepared || !x || !y) return fail(ONEBIT_ERR_ARGUMENT, "null operand pointer");
  if ((reinterpret_cast<uintptr_t>(x) & 15) != 0) return fail(ONEBIT_ERR_ARGUMENT, "x must be 16-byte aligned");
  const int kc_total = (k + onebit::kChunkK - 1) / onebit::kChunkK;
  const int compute_units = current_compute_units();
  const LinearPlan linear = plan_linear(m, tokens, k, compute_units);
  const LaunchPlan& plan = linear.launch;
  if ((size_t)k * 256 * 2 >= (size_t(1) << 32))
    return fail(ONEBIT_ERR_ARGUMENT, "the token-major form addresses x with 32-bit offsets inside a tile of 256 tokens: "
                                     "k = %d is beyond its limit of 8388607", k);
  if (linear.wide || plan.split_k_kernel) {
    onebit::SkinnyArgs args{};
    args.prep = static_cast<const uint8_t*>(prepared);
    args.b = static_cast<const _Float16*>(x);
    args.d = y;
    args.m = m; args.n = tokens; args.k = k;
    args.kc_total = kc_total;
    args.alpha = 1.f; args.beta = 0.f;
    args.d_f16 = y_dtype != ONEBIT_DTYPE_F32;
    args.bias = bias;
    args.bias_type = bias_dtype;
    args.bf16 = x_dtype == ONEBIT_DTYPE_BF16;
    args.x_f32 = x_dtype == ONEBIT_DTYPE_F32;
    DeviceLock lock;
    if (int rc = setup_skinny_split(args, linear.wide ? linear.wide_plan.splits : plan.splits, plan.splits, s, nullptr, lock);
        rc != ONEBIT_OK)
      return rc;
    args.tokens_per_group = linear.wide_plan.tokens;
    args.strips = linear.wide && wide_in_strips(m, tokens, k, linear.wide_plan, false, compute_units);
    ONEBIT_HIP(linear.wide ? onebit::launch_wide_tokens(args, linear.wide_plan.rows, s)
                           : onebit::launch_skinny_tokens(args, plan.rows_or_tile, s));
    return ONEBIT_OK;
  }
  switch (plan.rows_or_tile) {
    case onebit::kTile256x128w: case onebit::kTile128x128s: case onebit::kTile512x128w8: case onebit::kTile256x128w8:
    case onebit::kTile128x128w8: case onebit::kTile64x128: case onebit::kTile128x128k2: case onebit::kTile64x128k2:
    case onebit::kTile512x128m16: break;
    default:
      return fail(ONEBIT_ERR_ARGUMENT, "tile configuration %d has no token-major variant (4, 6, 9 ... 15 have)",
                  plan.rows_or_tile);
  }
  if (onebit::prepared_bytes(m, k) >= (size_t(1) << 32))
    return fail(ONEBIT_ERR_ARGUMENT,
                "the main kernel addresses the prepared operand with 32-bit offsets: m x k = %d x %d needs %zu bytes, "
                "the limit is 4 GiB (about 22.9e9 weights); split the weight by rows", m, k, onebit::prepared_bytes(m, k));
  onebit::GemmArgs args{};
  args.prep = static_cast<const uint8_t*>(prepared);
  args.b = static_cast<const _Float16*>(x);
  args.d = y;
  args.m = m; args.n = tokens; args.k = k;
  args.kc_total = kc_total;
  args.d_f16 = y_dtype != ONEBIT_DTYPE_F32;
  args.bias = bias;
  args.bias_type = bias_dtype;
  args.bf16 = x_dtype == ONEBIT_DTYPE_BF16;
  if (plan.splits > 1) {
    int device = 0;
    ONEBIT_HIP(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices) return fail(ONEBIT_ERR_ARGUMENT, "device ordinal %d not supported", device);
    DeviceState& st = g_dev[device];
    std::lock_guard<std::recursive_mutex> lock(st.mu);
    args.chunks_per_split = (kc_total + plan.splits - 1) / plan.splits;
    args.splits = full_splits(kc_total, plan.splits);
    Buffer& ws = st.split_ws[s];
    if (int rc = grow(&ws.ptr, &ws.bytes, (size_t)args.splits * m * tokens * sizeof(float), s); rc != ONEBIT_OK) return rc;
    args.split_ws = static_cast<float*>(ws.ptr);
    ONEBIT_HIP(onebit::launch_gemm_tokens(args, plan.rows_or_tile, s));
    return ONEBIT_OK;
  }
  ONEBIT_HIP(onebit::launch_gemm_tokens(args, plan.rows_or_tile, s));
  return ONEBIT_OK;
}

}  // namespace

extern "C" {

const char* onebit_sparse_last_error(void) { return g_last_error.c_str(); }

void onebit_sparse_set_tile_config(int tile_config) { g_tile_config = tile_config; }
void onebit_sparse_set_skinny_enabled(int enabled) { g_skinny_enabled = enabled ? 1 : 0; }
void onebit_sparse_set_skinny_rows(int rows) { g_skinny_rows = rows; }
void onebit_sparse_set_split_k(int splits) { g_split_k = splits; }
void onebit_sparse_set_pad_b(int enabled) { g_pad_b = enabled ? 1 : 0; }

int onebit_sparse_describe_call(int token_major, int m, int n, int k, int b_16_byte_aligned, int compute_units, int* plan) {
  g_last_error.clear();
  if (!plan) return fail(ONEBIT_ERR_ARGUMENT, "plan must not be null");
  if (compute_units < 0) return fail(ONEBIT_ERR_ARGUMENT, "compute_units must not be negative (got %d)", compute_units);
  if (int rc = check_shape(m, n, k)) return rc;
  const int units = compute_units ? compute_units : current_compute_units();
  LaunchPlan launch;
  WidePlan wide{};
  bool is_wide, pad_b = false;
  if (token_major) {
    const LinearPlan linear = plan_linear(m, n, k, units);
    launch = linear.launch;
    wide = linear.wide_plan;
    is_wide = linear.wide;
  } else {
    const ProductPlan product = plan_product(m, n, k, b_16_byte_aligned != 0, units, [] { return false; });
    launch = product.launch;
    wide = product.wide;
    pad_b = product.pad_b;
    is_wide = wide.rows != 0;
  }
  plan[0] = is_wide ? ONEBIT_KERNEL_WIDE : launch.split_k_kernel ? ONEBIT_KERNEL_SPLIT_K : ONEBIT_KERNEL_MAIN;
  plan[1] = is_wide ? wide.rows : launch.rows_or_tile;
  plan[2] = full_splits((k + onebit::kChunkK - 1) / onebit::kChunkK, is_wide ? wide.splits : launch.splits);
  plan[3] = pad_b;
  plan[4] = is_wide ? wide.tokens : 0;
  return ONEBIT_OK;
}

int onebit_sparse_describe_launch_for(int m, int n, int k, int b_16_byte_aligned, int compute_units, int* plan) {
  g_last_error.clear();
  if (!plan) return fail(ONEBIT_ERR_ARGUMENT, "plan must not be null");
  if (compute_units <= 0) return fail(ONEBIT_ERR_ARGUMENT, "compute_units must be positive (got %d)", compute_units);
  int call[5];
  if (int rc = onebit_sparse_describe_call(0, m, n, k, b_16_byte_aligned, compute_units, call); rc != ONEBIT_OK) return rc;
  std::copy(call, call + 4, plan);
  return ONEBIT_OK;
}

int onebit_sparse_describe_launch(int m, int n, int k, int b_16_byte_aligned, int* plan) {
  // the compute units of the current device, as the calls themselves plan; 256 when there is no usable device
  return onebit_sparse_describe_launch_for(m, n, k, b_16_byte_aligned, current_compute_units(), plan);
}

size_t onebit_sparse_prepared_bytes(int m, int k) {
  if (m <= 0 || k <= 0) return 0;
  return onebit::prepared_bytes(m, k);
}

int onebit_sparse_prepare(const void* a, const void* e, int m, int k, int meta_layout, void* prepared, void* stream) {
  g_last_error.clear();
  if (int rc = check_shape(m, 1, k)) return rc;
  if (!a || !e || !prepared) return fail(ONEBIT_ERR_ARGUMENT, "null operand pointer");
  if (meta_layout < ONEBIT_META_REFERENCE || meta_layout > ONEBIT_META_LOGICAL)
    return fail(ONEBIT_ERR_ARGUMENT, "unknown metadata layout %d", meta_layout);
  ONEBIT_HIP(onebit::launch_prepare(a, e, prepared, m, k, meta_layout, static_cast<hipStream_t>(stream)));
  return ONEBIT_OK;
}

int onebit_sparse_pack(const void* weight, int m, int k, int prune, void* a, void* e, int meta_layout, void* stream) {
  return onebit_sparse_pack_typed(weight, ONEBIT_DTYPE_F16, m, k, prune, a, e, meta_layout, stream);
}

int onebit_sparse_pack_typed(const void* weight, int weight_dtype, int m, int k, int prune, void* a, void* e,
                             int meta_layout, void* stream) {
  g_last_error.clear();
  if (int rc = check_shape(m, 1, k)) return rc;
  if (!weight || !a || !e) return fail(ONEBIT_ERR_ARGUMENT, "null operand pointer");
  if (weight_dtype < ONEBIT_DTYPE_F32 || weight_dtype > ONEBIT_DTYPE_BF16)
    return fail(ONEBIT_ERR_ARGUMENT, "weight dtype code must be 0 (fp32), 1 (fp16) or 2 (bf16), got %d", weight_dtype);
  if ((reinterpret_cast<uintptr_t>(weight) & 15) != 0)
    return fail(ONEBIT_ERR_ARGUMENT, "the dense weight must be 16-byte aligned");
  if ((reinterpret_cast<uintptr_t>(a) & 7) != 0 || (reinterpret_cast<uintptr_t>(e) & 1) != 0)
    return fail(ONEBIT_ERR_ARGUMENT, "a must be 8-byte aligned and e 2-byte aligned");
  if (meta_layout < ONEBIT_META_REFERENCE || meta_layout > ONEBIT_META_LOGICAL)
    return fail(ONEBIT_ERR_ARGUMENT, "unknown metadata layout %d", meta_layout);
  ONEBIT_HIP(onebit::launch_pack(weight, weight_dtype, a, e, m, k, prune, meta_layout, static_cast<hipStream_t>(stream)));
  return ONEBIT_OK;
}

int onebit_sparse_matmul_prepared(const void* prepared, const void* b, const void* c, void* d, int m, int n, int k,
                                  float alpha, float beta, int c_dtype, int d_dtype, void* stream) {
  g_last_error.clear();
  if (int rc = check_shape(m, n, k)) return rc;
  if (int rc = check_dtype(c_dtype, d_dtype)) return rc;
  return matmul_prepared_impl(prepared, b, c, d, m, n, k, alpha, beta, c_dtype, d_dtype, static_cast<hipStream_t>(stream));
}

int onebit_sparse_matmul_prepared_static(const void* prepared, const void* b, const void* c, void* d, int m, int n, int k,
                                         float alpha, float beta, int c_dtype, int d_dtype, void* stream) {
  g_last_error.clear();
  if (int rc = check_shape(m, n, k)) return rc;
  if (int rc = check_dtype(c_dtype, d_dtype)) return rc;
  int device = 0;
  ONEBIT_HIP(hipGetDevice(&device));
  if (device < 0 || device >= kMaxDevices) return fail(ONEBIT_ERR_ARGUMENT, "device ordinal %d not supported", device);
  DeviceState& st = g_dev[device];
  FixedScratch fixed{nullptr, kStaticScratchBytes};
  {
    std::lock_guard<std::recursive_mutex> lock(st.mu);
    if (!st.static_scratch) {
      // once per device, with that device current: the address of this device's copy of the array
      void* address = nullptr;
      ONEBIT_HIP(hipGetSymbolAddress(&address, HIP_SYMBOL(g_static_scratch)));
      if (!address) return fail(ONEBIT_ERR_HIP, "hipGetSymbolAddress returned a null address for the static workspace");
      st.static_scratch = static_cast<unsigned char*>(address);
    }
    fixed.base = st.static_scratch;
  }
  return matmul_prepared_impl(prepared, b, c, d, m, n, k, alpha, beta, c_dtype, d_dtype,
                              static_cast<hipStream_t>(stream), &fixed);
}

int onebit_sparse_linear_prepared(const void* prepared, const void* x, const void* bias, void* y, int tokens, int m,
                                  int k, int bias_dtype, int y_dtype, void* stream) {
  if (int rc = check_shape(m, tokens, k)) return rc;
  if (int rc = check_dtype(bias_dtype, y_dtype)) return rc;
  return onebit_sparse_linear_prepared_typed(prepared, x, bias, y, tokens, m, k, ONEBIT_DTYPE_F16, bias_dtype, y_dtype, stream);
}

int onebit_sparse_linear_prepared_typed(const void* prepared, const void* x, const void* bias, void* y, int tokens, int m,
                                        int k, int x_dtype, int bias_dtype, int y_dtype, void* stream) {
  g_last_error.clear();
  if (int rc = check_shape(m, tokens, k)) return rc;
  if (int rc = check_linear_dtypes(x_dtype, bias_dtype, y_dtype)) return rc;
  return linear_prepared_impl(prepared, x, bias, y, tokens, m, k, x_dtype, bias_dtype, y_dtype, static_cast<hipStream_t>(stream));
}

int onebit_sparse_linear_prepared_f32(const void* prepared, const void* x, const void* bias, void* y, int tokens, int m, int k,
                                      int bias_dtype, int y_dtype, void* stream) {
  g_last_error.clear();
  if (int rc = check_shape(m, tokens, k)) return rc;
  if (int rc = check_linear_dtypes(ONEBIT_DTYPE_F16, bias_dtype, y_dtype)) return rc;
  if (!takes_f32(tokens))
    return fail(ONEBIT_ERR_ARGUMENT, "fp32 activations are read by the kernel of up to %d tokens only (got %d): convert them to fp16",
                onebit::kSkinnyTokens, tokens);
  return linear_prepared_impl(prepared, x, bias, y, tokens, m, k, ONEBIT_DTYPE_F32, bias_dtype, y_dtype, static_cast<hipStream_t>(stream));
}

int onebit_sparse_linear_reads_f32(int tokens, int m, int k, void* stream) {
  g_last_error.clear();
  return check_shape(m, tokens, k) == ONEBIT_OK && takes_f32(tokens) &&
         reading_f32_is_faster(tokens, m, k, current_compute_units(), static_cast<hipStream_t>(stream));
}

int onebit_sparse_linear_prepared_grouped(const onebit_linear_problem* problems, int count, int tokens, int bias_dtype,
                                          int y_dtype, void* stream) {
  if (int rc = check_dtype(bias_dtype, y_dtype)) return rc;
  return onebit_sparse_linear_prepared_grouped_typed(problems, count, tokens, ONEBIT_DTYPE_F16, bias_dtype, y_dtype, stream);
}

int onebit_sparse_linear_prepared_grouped_typed(const onebit_linear_problem* problems, int count, int tokens, int x_dtype,
                                                int bias_dtype, int y_dtype, void* stream) {
  g_last_error.clear();
  if (!problems || count < 1) return fail(ONEBIT_ERR_ARGUMENT, "problems must point to at least one problem (count = %d)", count);
  if (int rc = check_linear_dtypes(x_dtype, bias_dtype, y_dtype)) return rc;
  for (int i = 0; i < count; ++i) {
    const onebit_linear_problem& q = problems[i];
    if (int rc = check_shape(q.m, tokens, q.k)) return rc;
    if (!q.prepared || !q.x || !q.y) return fail(ONEBIT_ERR_ARGUMENT, "null operand pointer in problem %d", i);
    if ((reinterpret_cast<uintptr_t>(q.x) & 15) != 0) return fail(ONEBIT_ERR_ARGUMENT, "x of problem %d must be 16-byte aligned", i);
    if ((size_t)q.k * 256 * 2 >= (size_t(1) << 32))
      return fail(ONEBIT_ERR_ARGUMENT, "the token-major form addresses x with 32-bit offsets inside a tile of 256 tokens: "
                                       "k = %d of problem %d is beyond its limit of 8388607", q.k, i);
  }
  // Beyond the split-K kernel's range of token counts, or with that kernel switched off, there is nothing to share:
  // one call of the single form per problem.
  if (tokens > onebit::kSkinnyMaxN || !g_skinny_enabled) {
    for (int i = 0; i < count; ++i) {
      const onebit_linear_problem& q = problems[i];
      if (int rc = onebit_sparse_linear_prepared_typed(q.prepared, q.x, q.bias, q.y, tokens, q.m, q.k, x_dtype, bias_dtype,
                                                       y_dtype, stream))
        return rc;
    }
    return ONEBIT_OK;
  }
  // Row group of the launch: as for one product with all the weight rows that does not split K.
  const int compute_units = current_compute_units();
  for (int first = 0; first < count; first += onebit::kSkinnyMaxGroup) {
    const int in_launch = std::min(count - first, onebit::kSkinnyMaxGroup);
    const bool wide = tokens > onebit::kSkinnyTokens;
    long groups[3] = {0, 0, 0};
    int longest_k = 0;
    for (int i = 0; i < in_launch; ++i) {
      const onebit_linear_problem& q = problems[first + i];
      for (int r = 0; r < 3; ++r) groups[r] += (q.m + kWideRows[r] - 1) / kWideRows[r];
      longest_k = std::max(longest_k, q.k);
    }
    WidePlan wide_plan{};
    if (wide) wide_plan = plan_wide(groups, 0.0, tokens, longest_k, false, 1, 1, compute_units);
    const int rows = wide ? wide_plan.rows
                     : g_skinny_rows > 0 ? g_skinny_rows
                     : single_round_rows(groups[0], groups[1], compute_units);
    if (rows != 32 && rows != 64 && rows != 128) return fail(ONEBIT_ERR_ARGUMENT, "row group %d: must be 32, 64 or 128", rows);
    onebit::SkinnyGroupArgs group{};
    group.count = in_launch;
    for (int i = 0; i < in_launch; ++i) {
      const onebit_linear_problem& q = problems[first + i];
      onebit::SkinnyArgs& args = group.problem[i];
      args.prep = static_cast<const uint8_t*>(q.prepared);
      args.b = static_cast<const _Float16*>(q.x);
      args.d = q.y;
      args.m = q.m; args.n = tokens; args.k = q.k;
      args.kc_total = (q.k + onebit::kChunkK - 1) / onebit::kChunkK;
      args.alpha = 1.f; args.beta = 0.f;
      args.d_f16 = y_dtype != ONEBIT_DTYPE_F32;
      args.bias = q.bias;
      args.bias_type = bias_dtype;
      args.bf16 = x_dtype == ONEBIT_DTYPE_BF16;
      args.tokens_per_group = wide_plan.tokens;
    }
    ONEBIT_HIP(wide ? onebit::launch_wide_tokens_group(group, rows, static_cast<hipStream_t>(stream))
                    : onebit::launch_skinny_group(group, rows, static_cast<hipStream_t>(stream)));
  }
  return ONEBIT_OK;
}

int onebit_sparse_matmul_ex(const void* a, const void* b, const void* c, void* d, const void* e, int m, int n, int k,
                            float alpha, float beta, int c_dtype, int d_dtype, int meta_layout, void* stream) {
  g_last_error.clear();
  if (int rc = check_shape(m, n, k)) return rc;
  if (int rc = check_dtype(c_dtype, d_dtype)) return rc;
  if (!a || !b || !d || !e) return fail(ONEBIT_ERR_ARGUMENT, "null operand pointer");
  if (beta != 0.f && !c) return fail(ONEBIT_ERR_ARGUMENT, "c must not be null when beta != 0");
  if (meta_layout < ONEBIT_META_REFERENCE || meta_layout > ONEBIT_META_LOGICAL)
    return fail(ONEBIT_ERR_ARGUMENT, "unknown metadata layout %d", meta_layout);
  hipStream_t s = static_cast<hipStream_t>(stream);
  int device = 0;
  ONEBIT_HIP(hipGetDevice(&device));
  if (device < 0 || device >= kMaxDevices) return fail(ONEBIT_ERR_HIP, "device index %d out of range", device);
  DeviceState& ds = g_dev[device];
  void* prep = nullptr;
  const int cache_entries = g_weight_cache_entries.load();
  // The lock is kept until the call's kernels are enqueued: a call from another thread that evicts this weight, or has to grow
  // this stream's buffer, frees the memory they read after a device synchronization, which then covers them.
  std::lock_guard<std::recursive_mutex> lock(ds.mu);
  if (cache_entries > 0) {
    for (auto& w : ds.weight_cache)
      if (w.a == a && w.e == e && w.m == m && w.k == k && w.layout == meta_layout) {
        w.last_use = ++ds.use_counter;
        if (w.stream != s) ONEBIT_HIP(hipStreamWaitEvent(s, w.ready, 0));  // its reorder kernel ran on another stream
        prep = w.prep;
        break;
      }
    if (!prep) {
      hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
      ONEBIT_HIP(hipStreamIsCapturing(s, &capture));
      if (capture != hipStreamCaptureStatusNone)
        return fail(ONEBIT_ERR_ARGUMENT, "a weight that is not in the cache yet cannot be added while the stream is "
                                         "being captured: run the call once outside the capture first");
      if ((int)ds.weight_cache.size() >= cache_entries) {  // evict the least recently used entry
        size_t victim = 0;
        for (size_t i = 1; i < ds.weight_cache.size(); ++i)
          if (ds.weight_cache[i].last_use < ds.weight_cache[victim].last_use) victim = i;
        ONEBIT_HIP(hipDeviceSynchronize());  // earlier work on any stream may still read it
        ONEBIT_HIP(hipFree(ds.weight_cache[victim].prep));
        ONEBIT_HIP(hipEventDestroy(ds.weight_cache[victim].ready));
        ds.weight_cache.erase(ds.weight_cache.begin() + victim);
      }
      DeviceState::CachedWeight w{a, e, m, k, meta_layout, nullptr, s, nullptr, ++ds.use_counter};
      ONEBIT_HIP(hipMalloc(&w.prep, onebit::prepared_bytes(m, k)));
      if (hipError_t st = hipEventCreateWithFlags(&w.ready, hipEventDisableTiming); st != hipSuccess) {
        (void)hipFree(w.prep);
        return fail(ONEBIT_ERR_HIP, "HIP error '%s' from hipEventCreateWithFlags", hipGetErrorString(st));
      }
      hipError_t st = onebit::launch_prepare(a, e, w.prep, m, k, meta_layout, s);
      if (st == hipSuccess) st = hipEventRecord(w.ready, s);
      if (st != hipSuccess) {
        (void)hipFree(w.prep);
        (void)hipEventDestroy(w.ready);
        return fail(ONEBIT_ERR_HIP, "HIP error '%s' while reordering a cached weight", hipGetErrorString(st));
      }
      ds.weight_cache.push_back(w);
      prep = w.prep;
    }
    return matmul_prepared_impl(prep, b, c, d, m, n, k, alpha, beta, c_dtype, d_dtype, s);
  }
  Buffer& own = ds.prep[s];
  if (int rc = grow(&own.ptr, &own.bytes, onebit::prepared_bytes(m, k), s)) return rc;
  prep = own.ptr;
  ONEBIT_HIP(onebit::launch_prepare(a, e, prep, m, k, meta_layout, s));
  return matmul_prepared_impl(prep, b, c, d, m, n, k, alpha, beta, c_dtype, d_dtype, s);
}

int onebit_sparse_clear_weight_cache(void) {
  g_last_error.clear();
  int previous = 0;
  const bool have_device = hipGetDevice(&previous) == hipSuccess;
  int rc = ONEBIT_OK;
  for (int device = 0; device < kMaxDevices; ++device) {
    DeviceState& ds = g_dev[device];
    std::lock_guard<std::recursive_mutex> lock(ds.mu);
    if (ds.weight_cache.empty()) continue;
    if (hipSetDevice(device) != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
      rc = fail(ONEBIT_ERR_HIP, "cannot synchronize device %d to clear its weight cache", device);
      continue;
    }
    for (auto& w : ds.weight_cache) {
      (void)hipFree(w.prep);
      (void)hipEventDestroy(w.ready);
    }
    ds.weight_cache.clear();
  }
  if (have_device) (void)hipSetDevice(previous);
  return rc;
}

int onebit_sparse_release_buffers(void) {
  g_last_error.clear();
  int previous = 0;
  const bool have_device = hipGetDevice(&previous) == hipSuccess;
  int rc = ONEBIT_OK;
  for (int device = 0; device < kMaxDevices; ++device) {
    DeviceState& ds = g_dev[device];
    std::lock_guard<std::recursive_mutex> lock(ds.mu);
    if (ds.prep.empty() && ds.split_ws.empty() && ds.b_pad.empty()) continue;
    if (hipSetDevice(device) != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
      rc = fail(ONEBIT_ERR_HIP, "cannot synchronize device %d to release its buffers", device);
      continue;
    }
    for (auto* buffers : {&ds.prep, &ds.split_ws, &ds.b_pad}) {
      for (auto& entry : *buffers)
        if (entry.second.ptr) (void)hipFree(entry.second.ptr);
      buffers->clear();
    }
  }
  if (have_device) (void)hipSetDevice(previous);
  return rc;
}

int onebit_sparse_set_weight_cache(int entries) {
  g_weight_cache_entries.store(entries > 0 ? entries : 0);
  return entries > 0 ? ONEBIT_OK : onebit_sparse_clear_weight_cache();
}

void onebit_sparse_matmul(void* a, void* b, void* c, void* d, void* e, int m, int n, int k) {
  const int rc = onebit_sparse_matmul_ex(a, b, c, d, e, m, n, k, 1.0f, 0.0f, ONEBIT_DTYPE_F32, ONEBIT_DTYPE_F32,
                                         ONEBIT_META_REFERENCE, nullptr);
  if (rc != ONEBIT_OK) {
    fprintf(stderr, "Got onebit_sparse_matmul error: %s\n", g_last_error.c_str());
    exit(EXIT_FAILURE);
  }
}

}  // extern "C"

// The reference header declares the entry point without extern "C" (include/onebit_sparse_tensor.h:5), so
// objects compiled against it reference the C++-mangled name; export that name as well.
void onebit_sparse_matmul_cxx_name(void* a, void* b, void* c, void* d, void* e, int m, int n, int k)
    __asm__("_Z20onebit_sparse_matmulPvS_S_S_S_iii");
__attribute__((visibility("default"))) void onebit_sparse_matmul_cxx_name(void* a, void* b, void* c, void* d, void* e,
                                                                          int m, int n, int k) {
  onebit_sparse_matmul(a, b, c, d, e, m, n, k);
}
