// Stand-in for the HIP runtime under the whole of libonebitmul: device memory is address ranges that nobody reads, a kernel launch is
// a record of the kernel's name. Which build of a kernel a call launches can then be checked without a GPU.
#include <hip/hip_runtime.h>

#include <cxxabi.h>

#include <map>
#include <string>

namespace {
std::map<const void*, std::string>& kernels() {  // host handle -> name; filled before main by the registration of the sources
  static std::map<const void*, std::string> names;
  return names;
}
std::string g_launched;  // names of the launches since the last reset, a line each
uintptr_t g_next = uintptr_t(1) << 40;
}  // namespace

extern "C" {

const char* stub_launched() { return g_launched.c_str(); }
void stub_reset() { g_launched.clear(); }

void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  int status = 0;
  char* demangled = abi::__cxa_demangle(name, nullptr, nullptr, &status);
  kernels()[host] = status == 0 ? demangled : name;
  free(demangled);
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void* function, dim3, dim3, void**, size_t, hipStream_t) {
  g_launched += kernels()[function] + "\n";
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipMalloc(void** ptr, size_t bytes) {
  *ptr = reinterpret_cast<void*>(g_next);
  g_next += (bytes + 4095) / 4096 * 4096;
  return hipSuccess;
}
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
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
  *status = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetSymbolAddress(void** address, const void*) { return hipMalloc(address, size_t(64) << 20); }
hipError_t hipEventCreate(hipEvent_t* event) {
  *event = nullptr;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* event, unsigned) { return hipEventCreate(event); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0.f;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }

}  // extern "C"
