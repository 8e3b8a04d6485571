// Device memory of the library and its copies to and from pageable host memory.
//
// hipMalloc + hipFree of a block of a few MB cost 30 to 250 us together (hipFree also waits for the
// device), and the loader, the top-k, the threshold compaction and the fixed-H learner need some
// ten such blocks per call: more than their kernels take.  Freed blocks of up to POOL_MAX_BLOCK
// bytes therefore stay with the library, at most POOL_CAP bytes of them, and serve later requests of
// the same size class (an eighth of a power of two).  They go back to the device when an allocation
// fails, when the free memory is asked for and on dnpeff_release_cached().
//
// A block is reused in the order of the library stream: whatever the library still has queued on
// it runs first.  (Blocks that the second stream touches live longer than any call.)  Callers who
// get or give back memory directly (dnpeff_dev_malloc / dnpeff_dev_free) may use other streams:
// those calls wait, as hipFree does.  One lock guards the lists.
#include "dnpeff_internal.hpp"

#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <utility>
#include <vector>

namespace dn {

constexpr size_t POOL_MAX_BLOCK = (size_t)256 << 20;
constexpr size_t POOL_CAP = (size_t)1 << 30;

struct pool_state {
  std::mutex lock;
  std::map<std::pair<int, size_t>, std::vector<void*>> idle;        // (device, class) -> blocks
  std::unordered_map<void*, std::pair<int, size_t>> live;           // blocks handed out
  size_t cached = 0;
};
static pool_state& pool() {
  static pool_state* p = new pool_state();  // (never destroyed: handles may outlive static destructors)
  return *p;
}

static size_t size_class(size_t bytes) {
  if (bytes <= 4096) return 4096;
  size_t g = 512;
  while (g * 16 <= bytes) g <<= 1;  // an eighth of the power of two below
  return (bytes + g - 1) / g * g;
}

static void trim_locked(pool_state& P) {
  for (auto& e : P.idle)
    for (void* p : e.second) (void)hipFree(p);
  P.idle.clear();
  P.cached = 0;
}

size_t pool_cached_bytes() {
  pool_state& P = pool();
  std::lock_guard<std::mutex> g(P.lock);
  return P.cached;
}

void pool_trim() {
  pool_state& P = pool();
  std::lock_guard<std::mutex> g(P.lock);
  trim_locked(P);
}

int device_alloc(void** out, size_t bytes, bool* reused) {
  *out = nullptr;
  if (reused) *reused = false;
  if (bytes == 0) bytes = 1;
  pool_state& P = pool();
  const bool pooled = bytes <= POOL_MAX_BLOCK;
  const size_t size = pooled ? size_class(bytes) : bytes;
  int dev = 0;
  if (pooled) {
    DN_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> g(P.lock);
    auto it = P.idle.find({dev, size});
    if (it != P.idle.end() && !it->second.empty()) {
      *out = it->second.back();
      it->second.pop_back();
      P.cached -= size;
      P.live[*out] = {dev, size};
      if (reused) *reused = true;
      return 0;
    }
  }
  hipError_t e = hipMalloc(out, size);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    pool_trim();
    e = hipMalloc(out, size);
  }
  if (e != hipSuccess) {
    set_error("hipMalloc of %zu bytes failed: %s", size, hipGetErrorString(e));
    return 1;
  }
  if (pooled) {
    std::lock_guard<std::mutex> g(P.lock);
    P.live[*out] = {dev, size};
  }
  return 0;
}

void device_release(void* p) {
  if (!p) return;
  pool_state& P = pool();
  {
    std::lock_guard<std::mutex> g(P.lock);
    auto it = P.live.find(p);
    if (it != P.live.end()) {
      const auto key = it->second;
      P.live.erase(it);
      if (P.cached + key.second <= POOL_CAP) {
        P.idle[key].push_back(p);
        P.cached += key.second;
        return;
      }
    }
  }
  (void)hipFree(p);
}

// ---------------------------------------------------------------------------
// Copies between pageable host memory and the device
//
// hipMemcpy takes pageable memory through its own staging on the calling thread: 29 GB/s up and 18
// GB/s down (less into memory that has not been touched yet) where the link carries 57 GB/s from
// pinned memory.  From STAGED_MIN bytes on, COPY_THREADS threads each move every COPY_THREADS-th
// piece through two pinned buffers of their own: the host copy (and the page faults of a fresh
// destination) of one piece runs beside the DMA of the others.  The copies are queued on the library
// stream (behind everything launched so far) and finished on return.
// ---------------------------------------------------------------------------
constexpr size_t STAGED_MIN = (size_t)4 << 20;
constexpr size_t STAGE_PIECE = (size_t)2 << 20;
constexpr int COPY_THREADS = 6;

struct stage_state {
  std::mutex lock;  // one staged copy at a time
  char* buf[COPY_THREADS][2] = {};
  hipEvent_t done[COPY_THREADS][2] = {};
};
static stage_state& stage() {
  static stage_state* s = new stage_state();
  return *s;
}

static bool stage_ready(stage_state& S) {
  for (int t = 0; t < COPY_THREADS; t++)
    for (int b = 0; b < 2; b++) {
      if (!S.buf[t][b] && hipHostMalloc((void**)&S.buf[t][b], STAGE_PIECE, hipHostMallocDefault) != hipSuccess) {
        S.buf[t][b] = nullptr;
        (void)hipGetLastError();
        return false;
      }
      if (!S.done[t][b] && hipEventCreateWithFlags(&S.done[t][b], hipEventDisableTiming) != hipSuccess) {
        S.done[t][b] = nullptr;
        (void)hipGetLastError();
        return false;
      }
    }
  return true;
}

static void stage_trim() {
  stage_state& S = stage();
  std::lock_guard<std::mutex> g(S.lock);
  for (int t = 0; t < COPY_THREADS; t++)
    for (int b = 0; b < 2; b++) {
      if (S.buf[t][b]) (void)hipHostFree(S.buf[t][b]);
      S.buf[t][b] = nullptr;
    }
}

template <bool UP>
static hipError_t staged_copy(char* dst, const char* src, size_t bytes) {
  stage_state& S = stage();
  std::lock_guard<std::mutex> g(S.lock);
  if (!stage_ready(S)) return hipMemcpy(dst, src, bytes, UP ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost);
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  hipStream_t st = stream();
  const size_t n_pieces = (bytes + STAGE_PIECE - 1) / STAGE_PIECE;
  std::atomic<int> failed{(int)hipSuccess};
  auto work = [&](int t) {
    hipError_t e = hipSetDevice(dev);
    size_t at[2] = {0, 0}, len[2] = {0, 0};  // downwards: the piece a buffer is receiving
    int k = 0;
    for (size_t p = (size_t)t; p < n_pieces && e == hipSuccess; p += COPY_THREADS, k++) {
      const int b = k & 1;
      const size_t off = p * STAGE_PIECE, n = off + STAGE_PIECE < bytes ? STAGE_PIECE : bytes - off;
      if (k >= 2) e = hipEventSynchronize(S.done[t][b]);
      if (e != hipSuccess) break;
      if (UP) {
        memcpy(S.buf[t][b], src + off, n);
        e = hipMemcpyAsync(dst + off, S.buf[t][b], n, hipMemcpyHostToDevice, st);
      } else {
        if (len[b]) memcpy(dst + at[b], S.buf[t][b], len[b]);
        e = hipMemcpyAsync(S.buf[t][b], src + off, n, hipMemcpyDeviceToHost, st);
        at[b] = off;
        len[b] = n;
      }
      if (e == hipSuccess) e = hipEventRecord(S.done[t][b], st);
    }
    // what is still on its way, the older piece first: the buffers are free again on return
    for (int i = k >= 2 ? k - 2 : 0; i < k; i++) {
      const int b = i & 1;
      const hipError_t es = hipEventSynchronize(S.done[t][b]);
      if (e == hipSuccess) e = es;
      if (!UP && e == hipSuccess) memcpy(dst + at[b], S.buf[t][b], len[b]);
    }
    if (e != hipSuccess) failed = (int)e;
  };
  const int n_threads = n_pieces < (size_t)COPY_THREADS ? (int)n_pieces : COPY_THREADS;
  std::vector<std::thread> helpers;
  for (int t = 1; t < n_threads; t++) helpers.emplace_back(work, t);
  work(0);
  for (std::thread& h : helpers) h.join();
  return (hipError_t)failed.load();
}

hipError_t copy_up(void* dst_dev, const void* src_host, size_t bytes) {
  if (bytes == 0) return hipSuccess;
  if (bytes < STAGED_MIN) return hipMemcpy(dst_dev, src_host, bytes, hipMemcpyHostToDevice);
  return staged_copy<true>((char*)dst_dev, (const char*)src_host, bytes);
}

hipError_t copy_down(void* dst_host, const void* src_dev, size_t bytes) {
  if (bytes == 0) return hipSuccess;
  if (bytes < STAGED_MIN) return hipMemcpy(dst_host, src_dev, bytes, hipMemcpyDeviceToHost);
  return staged_copy<false>((char*)dst_host, (const char*)src_dev, bytes);
}

// A few pinned words that kernels write results into (one stream synchronisation then replaces a
// device-to-host copy of some bytes and its round trip); one set per host thread.
int host_words(unsigned long long** out) {
  static thread_local unsigned long long* words = nullptr;
  if (!words) {
    DN_HIP(hipHostMalloc((void**)&words, 64 * sizeof(unsigned long long), hipHostMallocDefault));
  }
  *out = words;
  return 0;
}

}  // namespace dn

using namespace dn;

DN_API int dnpeff_release_cached(void) {
  clear_error();
  DN_HIP(hipStreamSynchronize(stream()));
  pool_trim();
  stage_trim();
  return 0;
}
