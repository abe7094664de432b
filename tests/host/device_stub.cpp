// Stand-in for the GPU under the host side of libonebitmul (csrc/onebit_capi.hip), which is linked against this file instead of
// the HIP runtime and the kernels: device memory is host memory that nobody reads, a launch is a record. What the host code
// decides (route, buffers, order of look-ups and launches between threads) can then be checked without a GPU.
//
// Allocations are address ranges of a reserved part of the address space; a launch that is handed one takes `stub_launch_us`
// before it looks at it and as long again while it uses it (two kernels, enqueued one after the other). Counted as violations: a
// range that was freed by then or is too small, partial sums or a padded copy that another thread's launch is using, an
// allocation freed during its use.
#include "onebit_launch.h"

#include <chrono>
#include <iterator>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <utility>

namespace {

constexpr uintptr_t kFirstAddress = uintptr_t(1) << 40;  // operands of the tests' calls lie below
std::mutex g_mu;
std::map<uintptr_t, size_t> g_memory;  // live allocations
std::map<uintptr_t, int> g_in_use;     // by launches
uintptr_t g_next = kFirstAddress;
std::string g_violation;               // the first one
int g_violations = 0, g_capturing = 0, g_launch_us = 0;
size_t g_allocated_total = 0;
thread_local hipError_t t_last_error = hipSuccess;  // of the thread's calls, until it is asked for, as in the HIP runtime

hipError_t last_error() { return std::exchange(t_last_error, hipSuccess); }

void violation(const char* what) {
  if (g_violations++ == 0) g_violation = what;
}

uintptr_t allocate(size_t bytes) {
  const uintptr_t at = g_next;
  g_next += (bytes + 4095) / 4096 * 4096;  // never handed out again
  g_memory[at] = bytes;
  g_allocated_total += bytes;
  return at;
}

struct Record {
  int kind, rows_or_tile, splits, columns_per_group, padded, m, n, k, strips;
};
Record g_last{};
enum Kind { kMain = 0, kSkinny = 1, kWide = 2 };

void pause() {
  if (g_launch_us > 0) std::this_thread::sleep_for(std::chrono::microseconds(g_launch_us));
}

// What a launch was handed; operands of the caller and null are skipped. shared: several launches may read it at a time.
struct Range {
  const void* at;
  size_t bytes;
  bool shared;
  bool owned() const { return reinterpret_cast<uintptr_t>(at) >= kFirstAddress; }
};

hipError_t launch(const Record& record, std::initializer_list<Range> ranges) {
  bool any = false;
  for (const Range& r : ranges) any = any || r.owned();
  if (any) pause();
  {
    std::lock_guard<std::mutex> lock(g_mu);
    g_last = record;
    for (const Range& r : ranges) {
      if (!r.owned()) continue;
      const uintptr_t at = reinterpret_cast<uintptr_t>(r.at);
      auto after = g_memory.upper_bound(at);
      if (after == g_memory.begin() || at + r.bytes > std::prev(after)->first + std::prev(after)->second)
        violation("a launch was given memory that had been freed or is too small");
      if (g_in_use[at]++ > 0 && !r.shared) violation("two launches used one buffer at the same time");
    }
  }
  if (any) pause();
  std::lock_guard<std::mutex> lock(g_mu);
  for (const Range& r : ranges)
    if (r.owned() && --g_in_use[reinterpret_cast<uintptr_t>(r.at)] == 0) g_in_use.erase(reinterpret_cast<uintptr_t>(r.at));
  return last_error();  // what the kernels' launchers return
}

template <class Args>
Range sums_of(const Args& a) {
  return Range{a.splits > 1 ? a.split_ws : nullptr, (size_t)a.splits * a.m * a.n * sizeof(float), false};
}
template <class Args>
Range weight_of(const Args& a) {
  return Range{a.prep, (size_t)((a.m + 31) / 32) * a.kc_total * 1536, true};
}

Record record_of(int kind, int rows_or_tile, const onebit::SkinnyArgs& a) {
  return Record{kind, rows_or_tile, a.splits, kind == kWide ? a.tokens_per_group : 0, 0, a.m, a.n, a.k, a.strips};
}

}  // namespace

namespace onebit {

hipError_t launch_prepare(const void*, const void*, void* prep, int m, int k, int, hipStream_t) {
  return launch(g_last, {Range{prep, (size_t)((m + 31) / 32) * ((k + 255) / 256) * 1536, false}});
}
hipError_t launch_pack(const void*, int, void*, void*, int, int, int, int, hipStream_t) { return hipSuccess; }
hipError_t launch_pad_b(const _Float16*, _Float16* dst, int k, int n, hipStream_t) {
  return launch(g_last, {Range{dst, (size_t)k * ((n + 7) / 8) * 16, false}});
}
hipError_t launch_gemm(GemmArgs a, int tile, hipStream_t) {
  return launch(Record{kMain, tile, a.splits, 0, a.b_pad != nullptr, a.m, a.n, a.k},
                {sums_of(a), Range{a.b_pad, (size_t)a.k * ((a.n + 7) / 8) * 16, false}, weight_of(a)});
}
hipError_t launch_gemm_tokens(GemmArgs a, int tile, hipStream_t) {
  return launch(Record{kMain, tile, a.splits, 0, 0, a.m, a.n, a.k}, {sums_of(a), weight_of(a)});
}
hipError_t launch_skinny(SkinnyArgs a, int rows, hipStream_t) { return launch(record_of(kSkinny, rows, a), {sums_of(a), weight_of(a)}); }
hipError_t launch_skinny_tokens(SkinnyArgs a, int rows, hipStream_t) {
  return launch(record_of(kSkinny, rows, a), {sums_of(a), weight_of(a)});
}
hipError_t launch_wide_tokens(SkinnyArgs a, int rows, hipStream_t) { return launch(record_of(kWide, rows, a), {sums_of(a), weight_of(a)}); }
hipError_t launch_wide(SkinnyArgs a, int rows, hipStream_t) {
  const Range b{a.b, (size_t)a.k * a.ldb * 2, false};  // owned if it is the padded copy
  Record r = record_of(kWide, rows, a);
  r.padded = b.owned();
  return launch(r, {sums_of(a), b, weight_of(a)});
}
hipError_t launch_skinny_group(SkinnyGroupArgs g, int rows, hipStream_t) {
  return launch(record_of(kSkinny, rows, g.problem[0]), {});
}
hipError_t launch_wide_tokens_group(SkinnyGroupArgs g, int rows, hipStream_t) {
  return launch(record_of(kWide, rows, g.problem[0]), {});
}

}  // namespace onebit

extern "C" {

int stub_violations() {
  std::lock_guard<std::mutex> lock(g_mu);
  return g_violations;
}
const char* stub_violation() { return g_violation.c_str(); }
void stub_set(int launch_us, int capturing) {  // capturing < 0: the question is refused
  std::lock_guard<std::mutex> lock(g_mu);
  g_launch_us = launch_us;
  g_capturing = capturing;
}
void stub_reset() {
  std::lock_guard<std::mutex> lock(g_mu);
  g_violations = 0;
  g_violation.clear();
  g_allocated_total = 0;
}
// the last launch: kind (0 main kernel, 1 skinny_kernel, 2 wide_kernel), rows or tile, splits, columns per group, padded copy
void stub_last_launch(int* out) {
  std::lock_guard<std::mutex> lock(g_mu);
  out[0] = g_last.kind;
  out[1] = g_last.rows_or_tile;
  out[2] = g_last.splits > 1 ? g_last.splits : 1;
  out[3] = g_last.padded;
  out[4] = g_last.columns_per_group;
}
// whether the last launch's grid is walked in strips of column groups
int stub_last_strips() {
  std::lock_guard<std::mutex> lock(g_mu);
  return g_last.strips;
}
size_t stub_allocated_bytes() {
  std::lock_guard<std::mutex> lock(g_mu);
  return g_allocated_total;
}

// ---- the HIP runtime as far as the host code calls it
hipError_t hipMalloc(void** ptr, size_t bytes) {
  std::lock_guard<std::mutex> lock(g_mu);
  *ptr = reinterpret_cast<void*>(allocate(bytes));
  return hipSuccess;
}
hipError_t hipFree(void* ptr) {
  std::lock_guard<std::mutex> lock(g_mu);
  const uintptr_t at = reinterpret_cast<uintptr_t>(ptr);
  if (g_in_use.count(at)) violation("an allocation was freed while a launch was using it");
  g_memory.erase(at);
  return hipSuccess;
}
hipError_t hipGetDevice(int* device) {
  *device = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t, int) {
  *value = 256;
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* status) {
  std::lock_guard<std::mutex> lock(g_mu);
  // the default stream while another one is captured
  if (g_capturing < 0) return t_last_error = hipErrorStreamCaptureImplicit;
  *status = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipGetLastError() { return last_error(); }
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetSymbolAddress(void** address, const void*) {
  static const uintptr_t scratch = allocate(size_t(64) << 20);
  *address = reinterpret_cast<void*>(scratch);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* event, unsigned) {
  *event = nullptr;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

}  // extern "C"
