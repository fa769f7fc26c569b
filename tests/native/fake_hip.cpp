// The HIP calls that csrc/runtime's dispatch makes, on the host and without a GPU: memory is malloc'd, a stream captures when the
// test says so, and a launch is handed to the test's callback instead of a device.  Linked with clusters.cpp and device_state.cpp
// into a library of the test's own.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <mutex>
#include <set>
#include <string>

#include "runtime_internal.hpp"

namespace {
std::mutex g_mu;
std::set<std::string> g_names;                         // a function handle is its name's address
std::set<hipStream_t> g_capturing;
typedef void (*launch_callback)(const char *name, uint32_t grid, uint32_t block, void *stream, void **args);
launch_callback g_callback = nullptr;
} // namespace

extern "C" {

__attribute__((visibility("default"))) void fake_set_launch_callback(launch_callback f) { g_callback = f; }
__attribute__((visibility("default"))) void fake_set_capturing(void *stream, int32_t on) {
  std::lock_guard<std::mutex> lock(g_mu);
  if (on)
    g_capturing.insert(static_cast<hipStream_t>(stream));
  else
    g_capturing.erase(static_cast<hipStream_t>(stream));
}
__attribute__((visibility("default"))) void fake_destroy_stream(void *stream) { mtrt_rt::forget_stream(static_cast<hipStream_t>(stream)); }

hipError_t hipGetDevice(int *device) { return *device = 0, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *prop, int) {
  std::memset(prop, 0, sizeof(*prop));
  std::strcpy(prop->gcnArchName, "gfx950");
  prop->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { return (*p = std::aligned_alloc(4096, (n + 4095) / 4096 * 4096)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t stream, hipStreamCaptureStatus *status) {
  std::lock_guard<std::mutex> lock(g_mu);
  *status = g_capturing.count(stream) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipModuleLoadData(hipModule_t *module, const void *) { return *module = reinterpret_cast<hipModule_t>(1), hipSuccess; }
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t *f, hipModule_t, const char *name) {
  std::lock_guard<std::mutex> lock(g_mu);
  *f = reinterpret_cast<hipFunction_t>(const_cast<char *>(g_names.insert(name).first->c_str()));
  return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned, unsigned, unsigned bx, unsigned, unsigned, unsigned, hipStream_t stream,
                                 void **args, void **) {
  if (g_callback)
    g_callback(reinterpret_cast<const char *>(f), gx, bx, stream, args);
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipGetLastError(void) { return hipSuccess; }

} // extern "C"

namespace mtrt_rt {
int32_t no_alloc_setup(DeviceState *, int) { return MTRT_OK; }
} // namespace mtrt_rt
