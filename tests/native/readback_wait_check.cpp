// Host-side check of readback.hip's pinned blocks: a call that fails after
// kernels were queued waits for the stream before its block can be lent
// again.  The HIP runtime is replaced by stubs that record what is queued.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../freeflow_amd/csrc/ff_internal.h"

static bool g_queued = false;      // a kernel was queued since the last wait
static bool g_fail_launch = false; // the next hipGetLastError reports an error
static bool g_dirty_free = false;  // host memory was freed with kernels queued

extern "C" {
char __hip_fatbin_stub;
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = *b = dim3(1);
  *s = 0;
  *st = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
  g_queued = true;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const bool f = g_fail_launch;
  g_fail_launch = false;
  return f ? hipErrorInvalidConfiguration : hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  g_queued = false;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  g_dirty_free = g_dirty_free || g_queued;
  std::free(p);
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return hipHostMalloc(p, n, 0); }
hipError_t hipFree(void* p) {
  g_queued = false;  // waits by itself
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
  g_queued = false;
  return hipSuccess;
}
}

namespace ff {
int hip_fail(hipError_t, const char*) { return FF_ERR_HIP; }
}  // namespace ff

static int bad = 0;
static void expect(bool ok, const char* what) {
  std::printf("%s: %s\n", what, ok ? "ok" : "WRONG");
  bad += ok ? 0 : 1;
}

int main() {
  ff::Domain d;
  float dev[4] = {}, host[4];
  const ff::Span span[1] = {{dev, host, sizeof(host)}};
  for (int domain = 0; domain < 2; domain++) {  // without and with idle blocks kept
    if (domain) ff::pinned_retain();
    expect(ff::read_spans(d, span, 1) == FF_OK && !g_queued, "gather");
    g_fail_launch = true;
    expect(ff::read_spans(d, span, 1) != FF_OK && !g_queued, "gather that reports an error");
    auto queue = [](ff::Domain&, void*) {
      g_queued = true;
      return (int)FF_OK;
    };
    auto queue_fail = [](ff::Domain&, void*) {
      g_queued = true;
      return (int)FF_ERR_HIP;
    };
    expect(ff::read_kernel_output(d, sizeof(host), host, queue) == FF_OK && !g_queued, "kernel output");
    expect(ff::read_kernel_output(d, sizeof(host), host, queue_fail) == FF_ERR_HIP && !g_queued,
           "kernel output whose launcher fails after a launch");
    expect(ff::read_kernel_output(d, (size_t)1 << 20, host, queue_fail) == FF_ERR_HIP && !g_queued,
           "the same without a block");
  }
  ff::pinned_release();
  expect(!g_dirty_free, "blocks freed idle");
  std::printf("wrong %d\n", bad);
  return bad ? 1 : 0;
}
