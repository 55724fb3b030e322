// readback.hip -- device results to host memory.
//
// A copy into pageable memory goes through the runtime's staging buffer: 15-30
// us for a few bytes, and for a flow field 5 (fresh pages) to 17 GB/s, because
// one thread copies behind one transfer.  Here kernels write results straight
// into pinned host memory (54 GB/s measured, as fast as the link) and the
// caller's threads copy on from there.

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "ff_internal.h"
#include "hermite.h"

namespace ff {

// ---------------------------------------------------------------- pinned blocks
// Blocks lent for one call.  A few idle ones of each size are kept while a
// domain lives (at most 4 x 256 KB and 8 x 4 MB for the process); calls on
// more threads than that allocate their own and free it again.
constexpr size_t kPinnedBytes[2] = {256u << 10, 4u << 20};
constexpr size_t kPinnedIdle[2] = {4, 8};

static std::mutex g_pinned_mu;
static std::vector<char*> g_pinned_idle[2];
static long long g_pinned_users = 0;

struct Slab {
  char* p;
  size_t used;
  int live;
};
static std::vector<Slab> g_slabs;

void pinned_retain() {
  std::lock_guard<std::mutex> lk(g_pinned_mu);
  for (int k = 0; k < 2; k++) g_pinned_idle[k].reserve(kPinnedIdle[k]);
  g_pinned_users++;
}

void pinned_release() {
  std::vector<char*> gone;
  {
    std::lock_guard<std::mutex> lk(g_pinned_mu);
    if (--g_pinned_users > 0) return;
    for (auto& v : g_pinned_idle) {
      gone.insert(gone.end(), v.begin(), v.end());
      v.clear();
    }
    for (auto& s : g_slabs) gone.push_back(s.p);  // empty: every domain is gone
    g_slabs.clear();
  }
  for (char* p : gone) (void)hipHostFree(p);
}

struct Pinned {
  const int kind;
  char* p = nullptr;  // null: no pinned memory left
  explicit Pinned(int k) : kind(k) {
    {
      std::lock_guard<std::mutex> lk(g_pinned_mu);
      if (!g_pinned_idle[kind].empty()) {
        p = g_pinned_idle[kind].back();
        g_pinned_idle[kind].pop_back();
        return;
      }
    }
    void* q = nullptr;
    if (hipHostMalloc(&q, kPinnedBytes[kind], hipHostMallocPortable) == hipSuccess) p = (char*)q;
    else (void)hipGetLastError();
  }
  Pinned(const Pinned&) = delete;
  ~Pinned() {
    if (!p) return;
    {
      std::lock_guard<std::mutex> lk(g_pinned_mu);
      if (g_pinned_users > 0 && g_pinned_idle[kind].size() < kPinnedIdle[kind]) {
        g_pinned_idle[kind].push_back(p);
        return;
      }
    }
    (void)hipHostFree(p);
  }
};

// Waits for the stream on every way out, errors too, before a block declared
// above it is lent again: kernels queued by a call that fails later still
// write the block.
struct StreamWait {
  const hipStream_t stream;
  bool done = false;
  hipError_t wait() {
    done = true;
    return hipStreamSynchronize(stream);
  }
  ~StreamWait() {
    if (!done) (void)hipStreamSynchronize(stream);
  }
};

// Small pinned pieces that live as long as their owner, cut from shared slabs
// (a pinned allocation of its own costs a domain 50-65 us).  A slab is given
// back when its last piece is freed; one empty slab is kept while a domain
// lives.
void* pinned_piece(size_t bytes) {
  bytes = (bytes + 63) & ~size_t(63);
  if (bytes > kPinnedPiece) return nullptr;
  std::lock_guard<std::mutex> lk(g_pinned_mu);
  Slab* s = nullptr;
  for (auto& x : g_slabs)
    if (x.used + bytes <= kPinnedBytes[0]) s = &x;
  if (!s) {
    void* q = nullptr;
    if (hipHostMalloc(&q, kPinnedBytes[0], hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_slabs.push_back({(char*)q, 0, 0});
    s = &g_slabs.back();
  }
  char* out = s->p + s->used;
  s->used += bytes;
  s->live++;
  return out;
}

void pinned_piece_free(void* p) {
  std::lock_guard<std::mutex> lk(g_pinned_mu);
  for (size_t k = 0; k < g_slabs.size(); k++) {
    Slab& s = g_slabs[k];
    if ((char*)p < s.p || (char*)p >= s.p + kPinnedBytes[0]) continue;
    if (--s.live > 0) return;
    s.used = 0;
    if (g_slabs.size() > 1) {
      (void)hipHostFree(s.p);
      g_slabs.erase(g_slabs.begin() + (long)k);
    }
    return;
  }
}

// ---------------------------------------------------------------- small results
constexpr int kMaxSpans = 4;
struct GatherArgs {
  const uint32_t* src[kMaxSpans];
  unsigned words[kMaxSpans], off[kMaxSpans];  // 4-byte words, at `off` of the block
  int n;
};

__global__ void __launch_bounds__(256) k_gather(GatherArgs a, uint32_t* __restrict__ out) {
  for (int s = 0; s < a.n; s++)
    for (unsigned k = blockIdx.x * 256 + threadIdx.x; k < a.words[s]; k += gridDim.x * 256) out[a.off[s] + k] = a.src[s][k];
}

int read_spans(Domain& d, const Span* spans, int n) {
  GatherArgs a{};
  size_t words = 0, largest = 0;
  for (int s = 0; s < n; s++) {
    a.src[s] = (const uint32_t*)spans[s].dev;
    a.words[s] = (unsigned)(spans[s].bytes / 4);
    a.off[s] = (unsigned)words;
    words += spans[s].bytes / 4;
    largest = std::max(largest, spans[s].bytes / 4);
  }
  a.n = n;
  if (!words) {
    FF_HIP(hipStreamSynchronize(d.stream));
    return FF_OK;
  }
  if (words * 4 <= kPinnedBytes[0]) {
    Pinned b(0);
    if (b.p) {
      StreamWait queued{d.stream};
      k_gather<<<(unsigned)std::min<size_t>(32, (largest + 255) / 256), 256, 0, d.stream>>>(a, (uint32_t*)b.p);
      FF_HIP(hipGetLastError());
      FF_HIP(queued.wait());
      for (int s = 0; s < n; s++)
        if (spans[s].bytes) std::memcpy(spans[s].host, b.p + (size_t)a.off[s] * 4, spans[s].bytes);
      return FF_OK;
    }
  }
  FF_HIP(hipStreamSynchronize(d.stream));
  for (int s = 0; s < n; s++)
    if (spans[s].bytes) FF_HIP(hipMemcpy(spans[s].host, spans[s].dev, spans[s].bytes, hipMemcpyDeviceToHost));
  return FF_OK;
}

int read_kernel_output(Domain& d, size_t bytes, void* out, int (*launch)(Domain&, void*)) {
  if (bytes <= kPinnedBytes[0]) {
    Pinned b(0);
    if (b.p) {
      StreamWait queued{d.stream};
      if (int rc = launch(d, b.p)) return rc;
      FF_HIP(queued.wait());
      std::memcpy(out, b.p, bytes);
      return FF_OK;
    }
  }
  void* tmp = nullptr;
  FF_HIP(hipMalloc(&tmp, std::max<size_t>(bytes, 16)));
  int rc = launch(d, tmp);
  if (!rc) {
    hipError_t e = hipStreamSynchronize(d.stream);
    if (e == hipSuccess) e = hipMemcpy(out, tmp, bytes, hipMemcpyDeviceToHost);
    if (e != hipSuccess) rc = hip_fail(e, "read results");
  }
  (void)hipFree(tmp);
  return rc;
}

// ---------------------------------------------------------------- flow fields
// Cells [c0, c0 + nc) of a moment buffer as records of NM floats at `out` (16
// byte aligned): transposed through LDS, so that the stores are whole
// 16-byte pieces of consecutive lanes (each store crosses the link by itself).
template <typename S, int DIM>
__global__ void __launch_bounds__(256) k_records(const S* __restrict__ soa, float* __restrict__ out, long long c0,
                                                 long long nc, size_t plane) {
  constexpr int NM = DIM == 2 ? 6 : 10;
  __shared__ __align__(16) float s[256 * NM];
  const long long b = (long long)blockIdx.x * 256;
  const int t = (int)threadIdx.x, m = (int)(nc - b < 256 ? nc - b : 256);
  if (t < m) {
#pragma unroll
    for (int q = 0; q < NM; q++) s[t * NM + q] = Store<S>::template load<DIM>(soa + q * plane + (c0 + b + t), q, plane);
  }
  __syncthreads();
  const int n = m * NM;
  float* o = out + b * NM;
  for (int k = 4 * t; k + 3 < n; k += 1024) *reinterpret_cast<float4*>(o + k) = *reinterpret_cast<const float4*>(s + k);
  for (int k = (n & ~3) + t; k < n; k += 256) o[k] = s[k];
}

static hipError_t launch_records(const Domain& d, const void* buf, float* out, long long c0, long long nc) {
  const unsigned g = (unsigned)((nc + 255) / 256);
#define FF_CV(S)                                                                                          \
  if (d.dim == 2) k_records<S, 2><<<g, 256, 0, d.stream>>>((const S*)buf, out, c0, nc, d.plane);          \
  else k_records<S, 3><<<g, 256, 0, d.stream>>>((const S*)buf, out, c0, nc, d.plane);
  if (d.storage == FF_STORAGE_F32) { FF_CV(float) }
  else if (d.storage == FF_STORAGE_F16) { FF_CV(__half) }
  else if (d.storage == FF_STORAGE_F16U) { FF_CV(h16u) }
  else { FF_CV(__hip_bfloat16) }
#undef FF_CV
  return hipGetLastError();
}

// A lane takes chunks of cells in turn until none is left: while a chunk's
// kernel fills one half of the lane's pinned block, the lane copies the other
// half's chunk into the caller's array.  One thread writes fresh pages at 13
// GB/s (27 warm), so a large field takes up to six lanes (eight or ten are no
// faster); a lane for every 1.5 MB pays for its thread (20-70 us).  Chunks of
// 2 MB for large fields (256x128x128: 168 MB in 3.8 ms, 4.5 with 1 MB, 5.1
// with 512 KB; 18.5 ms with one copy into pageable memory), of 512 KB below
// 16 MB, where a lane has few to overlap (61x47x39: 167 us against 210; 315).
constexpr size_t kHalf = kPinnedBytes[1] / 2, kHalfSmall = 512u << 10, kSmallField = 16u << 20;
constexpr int kMaxLanes = 6;
constexpr size_t kLaneBytes = 3u << 19;

static hipError_t moments_lane(const Domain& d, const void* buf, float* out, size_t half, std::atomic<long long>& next,
                               char* block) {
  hipError_t e = hipSetDevice(d.device);
  if (e != hipSuccess) return e;
  hipEvent_t ev[2] = {nullptr, nullptr};
  for (auto& v : ev)
    if (e == hipSuccess) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
  const long long per = (long long)(half / (d.nm * sizeof(float))) & ~255ll, chunks = (d.n + per - 1) / per;
  auto cells = [&](long long c) { return std::min(per, d.n - c * per); };
  long long flying = -1;  // chunk whose kernel fills the other half
  for (int k = 0; e == hipSuccess; k ^= 1) {
    const long long c = next.fetch_add(1);
    if (c < chunks) {
      e = launch_records(d, buf, (float*)(block + k * half), c * per, cells(c));
      if (e == hipSuccess) e = hipEventRecord(ev[k], d.stream);
    }
    if (flying >= 0 && e == hipSuccess) {
      e = hipEventSynchronize(ev[k ^ 1]);
      if (e == hipSuccess)
        std::memcpy(out + flying * per * d.nm, block + (k ^ 1) * half, (size_t)cells(flying) * d.nm * sizeof(float));
    }
    if (c >= chunks) break;
    flying = c;
  }
  if (e != hipSuccess) (void)hipStreamSynchronize(d.stream);  // no kernel may still write the block
  for (auto v : ev)
    if (v) (void)hipEventDestroy(v);
  return e;
}

int read_moments(Domain& d, const void* buf, float* out) {
  const size_t bytes = (size_t)d.n * d.nm * sizeof(float);
  const int want = (int)std::min<size_t>(kMaxLanes, std::max<size_t>(1, bytes / kLaneBytes));
  const size_t half = bytes < kSmallField ? kHalfSmall : kHalf;
  std::atomic<long long> next{0};
  hipError_t err[kMaxLanes] = {};
  {
    Pinned first(1);
    if (!first.p) {  // no pinned memory: through device memory, in one copy
      float* tmp = nullptr;
      FF_HIP(hipMalloc((void**)&tmp, bytes));
      hipError_t e = launch_records(d, buf, tmp, 0, d.n);
      if (e == hipSuccess) e = hipStreamSynchronize(d.stream);
      if (e == hipSuccess) e = hipMemcpy(out, tmp, bytes, hipMemcpyDeviceToHost);
      (void)hipFree(tmp);
      if (e != hipSuccess) return hip_fail(e, "download moments");
      return FF_OK;
    }
    std::thread lanes[kMaxLanes];
    for (int l = 1; l < want; l++) {
      try {
        lanes[l] = std::thread([&, l] {
          Pinned b(1);
          if (b.p) err[l] = moments_lane(d, buf, out, half, next, b.p);
        });
      } catch (...) {
        break;  // no more threads: the lanes that run take every chunk
      }
    }
    err[0] = moments_lane(d, buf, out, half, next, first.p);
    for (auto& t : lanes)
      if (t.joinable()) t.join();
  }
  for (const hipError_t e : err)
    if (e != hipSuccess) return hip_fail(e, "download moments");
  return FF_OK;
}

}  // namespace ff
