// A stand-in for the HIP runtime, linked with trueno_amd/csrc/trn_runtime.cpp by test_host_runtime.py: no GPU, kernels are
// launches in a list.  One device of 256 CUs; memory is addresses; a stream is captured or fails when the test says so.
#include <hip/hip_runtime_api.h>
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "../include/trueno_hip.h"

#define EXPORT extern "C" __attribute__((visibility("default")))

namespace {
struct Launch {
  std::string name;
  unsigned grid, block, lds;
  uint64_t stream, capture, args[5];
};
std::mutex g_lock;
std::vector<Launch> g_launches;
std::set<std::string> g_names;
std::map<uint64_t, size_t> g_memory;
std::map<uint64_t, unsigned long long> g_captures;
std::string g_fail;
uint64_t g_next = 0x100000000;
std::atomic<bool> g_record{true};
thread_local hipStreamCaptureMode t_mode = hipStreamCaptureModeGlobal;
bool refused() { return !g_captures.empty() && t_mode != hipStreamCaptureModeRelaxed; }
}  // namespace

EXPORT void fake_reset() {
  std::lock_guard<std::mutex> lock(g_lock);
  g_launches.clear();
  g_captures.clear();
  g_fail.clear();
}
EXPORT void fake_fail(const char* kernel) { g_fail = kernel; }      // launches of this kernel fail; "": none
EXPORT void fake_capture(uint64_t stream, unsigned long long id) {      // id 0: the capture ends
  std::lock_guard<std::mutex> lock(g_lock);
  if (id) g_captures[stream] = id;
  else g_captures.erase(stream);
}
EXPORT uint64_t fake_memory() {
  std::lock_guard<std::mutex> lock(g_lock);
  uint64_t sum = 0;
  for (auto& m : g_memory) sum += m.second;
  return sum;
}
EXPORT int fake_launches() { return int(g_launches.size()); }
EXPORT const char* fake_launch(int i, uint64_t* out) {      // out: grid, block, stream, capture, five arguments, LDS
  const Launch& l = g_launches[size_t(i)];
  out[0] = l.grid; out[1] = l.block; out[2] = l.stream; out[3] = l.capture;
  std::copy(l.args, l.args + 5, out + 4);
  out[9] = l.lds;
  return l.name.c_str();
}
// One thread issues a product over and over while another sets `key` to `value` or back to 0.  Of `rounds` changes, how many does the first thread not
// follow with a call that begins after the change has returned?
namespace { thread_local const void* t_last = nullptr; }
EXPORT int fake_tuning_race(const char* key, int value, uint32_t m, uint32_t n, uint32_t k, int rounds) {
  auto product = [&] {
    (void)trn_q4k_gemm(nullptr, 4096, 8192, 12288, m, n, k);
    return t_last;
  };
  const void* want[2];
  g_record = false;
  for (int s : {1, 0}) {
    (void)trn_set_tuning(key, s * value);
    want[s] = product();
  }
  if (want[0] == want[1]) return -1;
  std::atomic<int> done{0}, seen{0};
  std::thread setter([&] {
    for (int r = 1; r <= rounds; ++r) {
      while (seen.load() < r - 1) {}
      for (int spin = 0; spin < (r * 37) % 400; ++spin) (void)done.load();
      (void)trn_set_tuning(key, (r & 1) * value);
      done.store(r);
    }
  });
  int missed = 0;
  for (int r = 1; r <= rounds; ++r) {
    while (done.load() < r) (void)product();
    missed += product() != want[r & 1];
    seen.store(r);
  }
  setter.join();
  (void)trn_set_tuning(key, 0);
  g_record = true;
  return missed;
}

EXPORT hipError_t hipInit(unsigned) { return hipSuccess; }
EXPORT hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
EXPORT hipError_t hipSetDevice(int) { return hipSuccess; }
EXPORT hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
EXPORT hipError_t hipDeviceGet(hipDevice_t* d, int) { *d = 0; return hipSuccess; }
EXPORT hipError_t hipDeviceGetName(char* s, int n, hipDevice_t) { std::strncpy(s, "fake", size_t(n)); return hipSuccess; }
EXPORT hipError_t hipDeviceTotalMem(size_t* n, hipDevice_t) { *n = size_t(1) << 38; return hipSuccess; }
EXPORT hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) { *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeCooperativeLaunch; return hipSuccess; }
EXPORT hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  *p = hipDeviceProp_t{};
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
EXPORT hipError_t hipDeviceSynchronize() { return hipSuccess; }
EXPORT hipError_t hipGetLastError() { return hipSuccess; }
EXPORT const char* hipGetErrorName(hipError_t) { return "fake"; }
EXPORT const char* hipGetErrorString(hipError_t) { return "fake"; }
EXPORT hipError_t hipMemGetInfo(size_t* a, size_t* b) { *a = *b = size_t(1) << 38; return hipSuccess; }

EXPORT hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lock(g_lock);
  if (refused()) return hipErrorStreamCaptureUnsupported;
  *p = reinterpret_cast<void*>(g_next);
  g_memory[g_next] = n;
  g_next += (n + 4095u) / 4096u * 4096u;
  return hipSuccess;
}
EXPORT hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lock(g_lock);
  return g_memory.erase(reinterpret_cast<uint64_t>(p)) ? hipSuccess : hipErrorInvalidValue;
}
EXPORT hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = ::operator new(n); return hipSuccess; }
EXPORT hipError_t hipHostFree(void* p) { ::operator delete(p); return hipSuccess; }
EXPORT hipError_t hipHostGetDevicePointer(void** d, void* p, unsigned) { *d = p; return hipSuccess; }
EXPORT hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
EXPORT hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
EXPORT hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
EXPORT hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
EXPORT hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
EXPORT hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
EXPORT hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
EXPORT hipError_t hipModuleLoadData(hipModule_t* m, const void*) { *m = nullptr; return hipSuccess; }
EXPORT hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
EXPORT hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) {
  std::lock_guard<std::mutex> lock(g_lock);
  *f = reinterpret_cast<hipFunction_t>(const_cast<std::string*>(&*g_names.insert(name).first));
  return hipSuccess;
}
EXPORT hipError_t hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(int* n, hipFunction_t, int, size_t) { *n = 3; return hipSuccess; }
EXPORT hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned, unsigned, unsigned lds, hipStream_t s,
                                        void** args, void**) {
  const std::string& name = *reinterpret_cast<const std::string*>(f);
  t_last = f;
  if (!g_record) return hipSuccess;
  std::lock_guard<std::mutex> lock(g_lock);
  if (name == g_fail) return hipErrorLaunchFailure;
  if (uint64_t(gx) * bx >= uint64_t(1) << 32) return hipErrorInvalidConfiguration;
  Launch l{name, gx * gy * gz, bx, lds, reinterpret_cast<uint64_t>(s), 0, {}};
  auto capture = g_captures.find(l.stream);
  if (capture != g_captures.end()) l.capture = capture->second;
  if (name == "kq_fill_u32") std::memcpy(&l.args[0], args[0], 8);
  else for (int i = 0; i < 5 && name.find("gem") != std::string::npos; ++i) std::memcpy(&l.args[i], args[i], 8);      // (fifth: eight bytes of a u32 and what follows)
  g_launches.push_back(l);
  return hipSuccess;
}
EXPORT hipError_t hipModuleLaunchCooperativeKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz, unsigned lds,
                                                   hipStream_t s, void** args) {
  return hipModuleLaunchKernel(f, gx, gy, gz, bx, by, bz, lds, s, args, nullptr);
}
EXPORT hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = reinterpret_cast<hipStream_t>(g_next += 4096); return hipSuccess; }
EXPORT hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
EXPORT hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
EXPORT hipError_t hipStreamGetCaptureInfo(hipStream_t s, hipStreamCaptureStatus* status, unsigned long long* id) {
  std::lock_guard<std::mutex> lock(g_lock);
  auto it = g_captures.find(reinterpret_cast<uint64_t>(s));
  *status = it == g_captures.end() ? hipStreamCaptureStatusNone : hipStreamCaptureStatusActive;
  if (id) *id = it == g_captures.end() ? 0 : it->second;
  return hipSuccess;
}
EXPORT hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* status) { return hipStreamGetCaptureInfo(s, status, nullptr); }
EXPORT hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* mode) { std::swap(*mode, t_mode); return hipSuccess; }

// trn_noalloc.hip's
extern "C" hipError_t trn_noalloc_scratch_setup(int) { return hipSuccess; }
extern "C" uint64_t trn_noalloc_scratch(int, size_t* bytes) { *bytes = (size_t(16) << 20) + 65536; return 0x10000; }
extern "C" uint64_t trn_noalloc_workspace(int, size_t* bytes) { *bytes = size_t(256) << 20; return 0x20000000; }
