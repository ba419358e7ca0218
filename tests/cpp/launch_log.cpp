// Stand-in for the HIP runtime functions that libprichs_hip.so calls, for CPU
// tests of what the library launches.  Loaded before the library with
// RTLD_GLOBAL, it answers as a machine of eight 256-CU GPUs: device memory is
// host memory, and instead of running a kernel it notes its name, grid,
// workgroup, dynamic LDS and device.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <cxxabi.h>
#include <map>
#include <string>
#include <vector>

namespace {
struct Config {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
std::map<const void *, std::string> &names() {
  static std::map<const void *, std::string> m;
  return m;
}
std::vector<Config> g_configs;
std::string g_log, g_text;
int g_device = 0;
hipError_t g_error = hipSuccess;

std::string demangled(const std::string &s) {
  int status = 0;
  char *d = abi::__cxa_demangle(s.c_str(), nullptr, nullptr, &status);
  const std::string out = status == 0 ? d : s;
  std::free(d);
  return out;
}
}  // namespace

extern "C" {
// The log so far, one line per event; cleared by the call.
const char *launch_log_take() {
  g_text.swap(g_log);
  g_log.clear();
  return g_text.c_str();
}

void **__hipRegisterFatBinary(const void *) {
  static void *handle = nullptr;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
  names()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
  g_configs.push_back({grid, block, lds, stream});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream) {
  const Config c = g_configs.back();
  g_configs.pop_back();
  *grid = c.grid, *block = c.block, *lds = c.lds, *stream = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 g, dim3 b, void **, size_t lds, hipStream_t) {
  // The runtime's limit on the threads of a launch in each dimension.
  if ((unsigned long long)g.x * b.x > 0xffffffffull || g.y > 65535u * 65535u || g.x == 0)
    return g_error = hipErrorInvalidConfiguration;
  g_log += "launch\t" + demangled(names()[fn]) + "\t" + names()[fn] + "\t" + std::to_string(g.x) +
           "\t" + std::to_string(g.y) + "\t" + std::to_string(g.z) + "\t" + std::to_string(b.x) +
           "\t" + std::to_string(lds) + "\t" + std::to_string(g_device) + "\n";
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *fn, hipFuncAttribute, int value) {
  g_log += "attribute\t" + demangled(names()[fn]) + "\t" + std::to_string(value) + "\t" +
           std::to_string(g_device) + "\n";
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_error;
  g_error = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "launch_log error"; }

hipError_t hipGetDevice(int *d) {
  *d = g_device;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  g_device = d;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) {
  *p = std::aligned_alloc(256, (n + 255) / 256 * 256);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidSymbol; }
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 0.0f;
  return hipSuccess;
}
}  // extern "C"
