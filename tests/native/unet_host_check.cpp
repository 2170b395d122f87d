// CPU check of the network's host code (csrc/fs_unet.hip, compiled for the
// host alone) against a HIP runtime of stand-ins: device memory is addresses
// that nothing reads, launches and copies are noted, and any call can be made
// to fail.  Built and run by tests/test_unet_host.py.
//   batches H W max_batch   loss_grad of every batch 1..max_batch: "batch
//                           status" of those that fail, then the number tried
//   failures H W batch      loss_grad with its first, second, ... runtime call
//                           failing: "call name streams" of those that return
//                           with copies of the caller's arrays not waited for,
//                           then the number of calls
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "fastscape.h"

namespace {
long g_calls = 0, g_fail = 0;        // runtime calls so far; the one to fail (0: none)
bool g_failed = false;
std::string g_name;                  // of the failed call
hipError_t g_last = hipSuccess;
uintptr_t g_next = 1ull << 60;       // next device address
std::map<hipStream_t, int> g_copies; // host copies not waited for, by stream

hipError_t call(const char *name) {
  if (g_fail && ++g_calls == g_fail) {
    g_failed = true;
    g_name = name;
    return g_last = hipErrorUnknown;
  }
  return hipSuccess;
}
bool on_device(const void *p) { return reinterpret_cast<uintptr_t>(p) >= 1ull << 60; }
hipError_t give(void **p, size_t n) {
  *p = reinterpret_cast<void *>(g_next);
  g_next += (n + 4095) / 4096 * 4096;
  return hipSuccess;
}
template <class T>
hipError_t handle(T *h) {
  void *p;
  give(&p, 1);
  *h = static_cast<T>(p);
  return hipSuccess;
}
}  // namespace

#define STAND_IN(name)              \
  do {                              \
    const hipError_t e = call(name); \
    if (e != hipSuccess) return e;  \
  } while (0)

extern "C" {
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { STAND_IN("hipSetDevice"); return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return give(p, n); }
hipError_t hipFree(void *) { return hipSuccess; }
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t, hipMemcpyKind, hipStream_t st) {
  STAND_IN("hipMemcpyAsync");
  if (!on_device(d) || !on_device(s)) g_copies[st]++;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  // a wait that fails waits all the same: nothing more can be asked of a caller
  g_copies.erase(s);
  STAND_IN("hipStreamSynchronize");
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
  STAND_IN("hipStreamWaitEvent");
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { STAND_IN("hipEventRecord"); return hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "made to fail"; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
  STAND_IN("hipLaunchKernel");
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s) {
  *g = *b = dim3(1);
  *n = 0;
  *s = nullptr;
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *,
                           void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}

int main(int argc, char **argv) {
  if (argc < 5) return 2;
  const int H = std::atoi(argv[2]), W = std::atoi(argv[3]), B = std::atoi(argv[4]);
  fs_unet *u = nullptr;
  if (fs_unet_create(H, W, B, 1, 0, &u) != FS_OK) return 3;
  size_t n = 0;
  fs_unet_param_count(u, &n);
  // the caller's arrays: host addresses that nothing reads either
  float host[8] = {};
  const float *terrain = host, *params = host + 1, *target = host + 2;
  float *loss = host + 3, *grad = host + 4;
  if (!std::strcmp(argv[1], "batches")) {
    for (int b = 1; b <= B; b++) {
      const int st = fs_unet_loss_grad(u, terrain, params, target, b, loss, grad, n);
      if (st != FS_OK) std::printf("%d %d\n", b, st);
    }
    std::printf("%d\n", B);
  } else {
    for (g_fail = 1;; g_fail++) {
      g_calls = 0;
      g_failed = false;
      g_last = hipSuccess;
      g_copies.clear();
      const int st = fs_unet_loss_grad(u, terrain, params, target, B, loss, grad, n);
      if (!g_failed) break;
      if (st == FS_OK) std::printf("%ld %s status\n", g_fail, g_name.c_str());
      if (!g_copies.empty())
        std::printf("%ld %s %zu\n", g_fail, g_name.c_str(), g_copies.size());
    }
    std::printf("%ld\n", g_fail - 1);
  }
  g_fail = 0;
  fs_unet_destroy(u);
  return 0;
}
