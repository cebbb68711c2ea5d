// A HIP runtime for host tests of the library's launch code: no device, every
// call that reaches it is logged. Loaded with RTLD_GLOBAL before the library,
// its functions come before the real runtime's. Built by test_workspaces_host.py.
#include <hip/hip_runtime_api.h>

#include <stdint.h>
#include <string.h>
#include <unistd.h>

#include <atomic>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace {
std::mutex mu;
std::map<const void *, std::string> names;      // host stub -> kernel
std::map<void *, bool> capturing;               // stream -> being captured
bool global_capture = false;                    // some thread captures in global mode
useconds_t launch_us = 0;                       // pause after each launch
std::string text;
uintptr_t next_ptr = (uintptr_t)1 << 46;
std::map<std::thread::id, int> threads;         // in order of their first event
std::atomic<int> module{0};
thread_local hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
thread_local hipError_t last = hipSuccess;
struct Config {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
thread_local std::vector<Config> configs;

void event(const std::string &what) {
  std::lock_guard<std::mutex> lk(mu);
  const int id = threads.emplace(std::this_thread::get_id(), (int)threads.size()).first->second;
  text += std::to_string(id) + " " + what + "\n";
}
}  // namespace

extern "C" {

const char *fake_log(void) { return text.c_str(); }
void fake_reset(void) {
  std::lock_guard<std::mutex> lk(mu);
  text.clear();
  threads.clear();
}
void fake_pause(int us) { launch_us = us; }
void fake_capture(void *stream, int on) { capturing[stream] = on; }
void fake_global_capture(int on) { global_capture = on; }

void **__hipRegisterFatBinary(const void *) { return (void **)&module; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, dim3 *, dim3 *, int *) {
  names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
  configs.push_back(Config{grid, block, lds, stream});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream) {
  const Config c = configs.back();
  configs.pop_back();
  *grid = c.grid;
  *block = c.block;
  *lds = c.lds;
  *stream = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 grid, dim3, void **, size_t, hipStream_t stream) {
  event("launch " + std::to_string((uintptr_t)stream) + " " +
        std::to_string((uint64_t)grid.x * grid.y * grid.z) + " " + names[fn]);
  if (launch_us) usleep(launch_us);
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = (void *)((uintptr_t)1 << 45); return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *out) {
  *out = capturing[(void *)s] ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) {
  std::swap(mode, *m);
  return hipSuccess;
}
// While a thread captures in global mode, a call that synchronises is refused
// to every thread that has not relaxed its own mode.
hipError_t hipMalloc(void **p, size_t bytes) {
  if (global_capture && mode != hipStreamCaptureModeRelaxed) {
    event("refused " + std::to_string(bytes));
    return last = hipErrorStreamCaptureUnsupported;
  }
  event("malloc " + std::to_string(bytes));
  std::lock_guard<std::mutex> lk(mu);
  *p = (void *)next_ptr;
  next_ptr += (bytes + 4095) & ~(size_t)4095;
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *, int, size_t bytes, hipStream_t) {
  event("memset " + std::to_string(bytes));
  return hipSuccess;
}

}  // extern "C"
