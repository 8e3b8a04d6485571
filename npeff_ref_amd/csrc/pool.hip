// Device memory of the library and its copies to and from pageable host memory.
//
// hipMalloc + hipFree of a block of a few MB cost 30 to 250 us together (hipFree also waits for the
// device), and the loader, the top-k, the threshold compaction and the fixed-H learner need some
// ten such blocks per call: more than their kernels take.  Freed blocks of up to POOL_MAX_BLOCK
// bytes therefore stay with the library, at most POOL_CAP bytes of them, and serve later requests of
// the same size class (an eighth of a power of two).  They go back to the device when an allocation
// fails, when the free memory is asked for and on dnpeff_release_cached().  Other allocators of the
// process cannot ask for them: more than POOL_LOW bytes are kept only while a sixteenth of the device is
// free, as last seen at most 0.1 s ago and since the last large block (hipMemGetInfo waits for kernels
// under way: asked at every release it added 20 to 80 us to the calls of the fixed-H learner and the top-k).
//
// A block is reused in the order of the library stream: whatever the library still has queued on
// it runs first.  (Blocks that the second stream touches live longer than any call.)  Callers who
// get or give back memory directly (dnpeff_dev_malloc / dnpeff_dev_free) may use other streams:
// those calls wait, as hipFree does.  One lock guards the lists.
#include "dnpeff_internal.hpp"
#include "host_parts.hpp"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

namespace dn {

constexpr size_t POOL_MAX_BLOCK = (size_t)256 << 20;
constexpr size_t POOL_CAP = (size_t)1 << 30;
constexpr size_t POOL_LOW = (size_t)64 << 20;

struct pool_state {
  std::mutex lock;
  std::map<std::pair<int, size_t>, std::vector<void*>> idle;        // (device, class) -> blocks
  std::unordered_map<void*, std::pair<int, size_t>> live;           // blocks handed out
  size_t cached = 0;
  bool asked = false, is_short = false;  // whether the device was nearly full, and when that was looked up
  std::chrono::steady_clock::time_point asked_at;
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

static bool memory_is_short(pool_state& P) {
  const auto now = std::chrono::steady_clock::now();
  if (!P.asked || now - P.asked_at > std::chrono::milliseconds(100)) {
    size_t free_b = 0, total_b = 0;
    P.is_short = hipMemGetInfo(&free_b, &total_b) != hipSuccess || free_b < total_b / 16;
    P.asked = true;
    P.asked_at = now;
  }
  return P.is_short;
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
    (void)hipGetLastError();  // (reported here: not by the next launch of whoever does without the block)
    set_error("hipMalloc of %zu bytes failed: %s", size, hipGetErrorString(e));
    return 1;
  }
  std::lock_guard<std::mutex> g(P.lock);
  if (pooled) P.live[*out] = {dev, size};
  else P.asked = false;
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
      bool keep = P.cached + key.second <= POOL_CAP;
      if (keep && P.cached + key.second > POOL_LOW && memory_is_short(P)) {
        trim_locked(P);
        keep = false;
      }
      if (keep) {
        try {
          P.idle[key].push_back(p);
          P.cached += key.second;
          return;
        } catch (...) {  // (no memory to note it: back to the device)
        }
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
// destination) of one piece runs beside the transfer of the others.  A transfer is a kernel that reads or
// writes the pinned buffer (a piece on the copy engines waits 14 us for its turn), the threads alternate
// between two streams, so that one piece's completion is not in the way of the next, and several arrays go
// as one run of pieces.  The copies wait for everything launched on the library stream so far and are
// finished on return.  131 MB in two arrays: 2.6 ms up and 2.9 ms
// down, 3.7 and 3.4 ms piece by piece on the copy engines (64 workgroups the same, 128 slower).
// ---------------------------------------------------------------------------
constexpr size_t STAGED_MIN = (size_t)4 << 20;
constexpr size_t STAGE_PIECE = (size_t)2 << 20;
constexpr int COPY_THREADS = 8;
constexpr int COPY_STREAMS = 2;
constexpr int COPY_WGS = 32;

struct stage_state {
  std::mutex lock;  // one staged copy at a time
  int dev = -1;
  char* buf[COPY_THREADS][2] = {};
  hipEvent_t done[COPY_THREADS][2] = {};
  hipEvent_t before = nullptr;  // what the library stream had to do
  hipStream_t st[COPY_STREAMS] = {};
};
static stage_state& stage() {
  static stage_state* s = new stage_state();
  return *s;
}

static void stage_free(stage_state& S) {
  for (int t = 0; t < COPY_THREADS; t++)
    for (int b = 0; b < 2; b++) {
      if (S.buf[t][b]) (void)hipHostFree(S.buf[t][b]);
      if (S.done[t][b]) (void)hipEventDestroy(S.done[t][b]);
      S.buf[t][b] = nullptr;
      S.done[t][b] = nullptr;
    }
  for (hipStream_t& st : S.st) {
    if (st) (void)hipStreamDestroy(st);
    st = nullptr;
  }
  if (S.before) (void)hipEventDestroy(S.before);
  S.before = nullptr;
  S.dev = -1;
}

static bool stage_ready(stage_state& S, int dev) {
  if (S.dev == dev) return true;
  stage_free(S);
  bool ok = hipEventCreateWithFlags(&S.before, hipEventDisableTiming) == hipSuccess;
  for (int t = 0; t < COPY_THREADS && ok; t++)
    for (int b = 0; b < 2 && ok; b++)
      ok = hipHostMalloc((void**)&S.buf[t][b], STAGE_PIECE, hipHostMallocDefault) == hipSuccess &&
           hipEventCreateWithFlags(&S.done[t][b], hipEventDisableTiming) == hipSuccess;
  for (int q = 0; q < COPY_STREAMS && ok; q++) ok = hipStreamCreateWithFlags(&S.st[q], hipStreamNonBlocking) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    stage_free(S);
    return false;
  }
  S.dev = dev;
  return true;
}

static void stage_trim() {
  stage_state& S = stage();
  std::lock_guard<std::mutex> g(S.lock);
  stage_free(S);
}

__global__ void __launch_bounds__(256) k_copy_piece(const uint4* __restrict__ src, uint4* __restrict__ dst, int n) {
  for (int at = blockIdx.x * 1024 + threadIdx.x; at < n; at += gridDim.x * 1024) {
    uint4 v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) v[u] = src[at + 256 * u < n ? at + 256 * u : n - 1];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (at + 256 * u < n) dst[at + 256 * u] = v[u];
  }
}

static hipError_t piece_copy(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t st) {
  if (n % 16 != 0 || (uintptr_t)dst % 16 != 0 || (uintptr_t)src % 16 != 0) return hipMemcpyAsync(dst, src, n, kind, st);
  const int quads = (int)(n / 16), wgs = (quads + 1023) / 1024;
  hipLaunchKernelGGL(k_copy_piece, dim3(wgs < COPY_WGS ? wgs : COPY_WGS), dim3(256), 0, st, (const uint4*)src,
                     (uint4*)dst, quads);
  return hipGetLastError();
}

template <bool UP>
static hipError_t staged_copy(const copy_part* parts, int n_parts) {
  stage_state& S = stage();
  std::lock_guard<std::mutex> g(S.lock);
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (!stage_ready(S, dev)) {
    for (int q = 0; q < n_parts && e == hipSuccess; q++)
      e = hipMemcpy(parts[q].dst, parts[q].src, parts[q].bytes, UP ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost);
    return e;
  }
  e = hipEventRecord(S.before, stream());
  for (int q = 0; q < COPY_STREAMS && e == hipSuccess; q++) e = hipStreamWaitEvent(S.st[q], S.before, 0);
  if (e != hipSuccess) return e;
  size_t n_pieces = 0;
  for (int q = 0; q < n_parts; q++) n_pieces += (parts[q].bytes + STAGE_PIECE - 1) / STAGE_PIECE;
  std::atomic<int> failed{(int)hipSuccess};
  auto work = [&](int t) {
    hipError_t e = hipSetDevice(dev);
    hipStream_t st = S.st[t % COPY_STREAMS];
    char* to[2] = {};  // downwards: where the piece goes that a buffer is receiving
    size_t len[2] = {0, 0};
    int k = 0, part = 0;
    size_t first = 0;  // the part's first piece
    for (size_t p = (size_t)t; p < n_pieces && e == hipSuccess; p += COPY_THREADS, k++) {
      for (;; part++) {
        const size_t of_part = (parts[part].bytes + STAGE_PIECE - 1) / STAGE_PIECE;
        if (p < first + of_part) break;
        first += of_part;
      }
      const size_t off = (p - first) * STAGE_PIECE, left = parts[part].bytes - off;
      const size_t n = left < STAGE_PIECE ? left : STAGE_PIECE;
      const char* src = (const char*)parts[part].src + off;
      char* dst = (char*)parts[part].dst + off;
      const int b = k & 1;
      if (k >= 2) e = hipEventSynchronize(S.done[t][b]);
      if (e != hipSuccess) break;
      if (UP) {
        memcpy(S.buf[t][b], src, n);
        e = piece_copy(dst, S.buf[t][b], n, hipMemcpyHostToDevice, st);
      } else {
        if (len[b]) memcpy(to[b], S.buf[t][b], len[b]);
        e = piece_copy(S.buf[t][b], src, n, hipMemcpyDeviceToHost, st);
        to[b] = dst;
        len[b] = n;
      }
      if (e == hipSuccess) e = hipEventRecord(S.done[t][b], st);
      if (!UP && e == hipSuccess) fetch_pages(dst, n);
    }
    // what is still on its way, the older piece first: the buffers are free again on return
    for (int i = k >= 2 ? k - 2 : 0; i < k; i++) {
      const int b = i & 1;
      const hipError_t es = hipEventSynchronize(S.done[t][b]);
      if (e == hipSuccess) e = es;
      if (!UP && e == hipSuccess) memcpy(to[b], S.buf[t][b], len[b]);
    }
    if (e != hipSuccess) failed = (int)e;
  };
  const int n_threads = n_pieces < (size_t)COPY_THREADS ? (int)n_pieces : COPY_THREADS;
  run_shares(n_threads, work, [](auto f) { return std::thread(f); });
  return (hipError_t)failed.load();
}


// Smaller copies go through one of a few pinned buffers, which kernels read and write.
// (hipMemcpy of a few bytes from or to pageable memory takes 30 to 70 us here, and now and then
// milliseconds for some MB; 15 us this way.  hipMemcpyAsync from and to the buffer is longer too, and in one process of some
// twenty took 120 us more for every copy down.)
constexpr size_t BOUNCE_HALF = (size_t)1 << 20;
constexpr int BOUNCE_PIECES = pinned_buf::EVENTS;  // upwards
constexpr size_t BOUNCE_KERNEL = 16384;
constexpr size_t BOUNCE_KEPT = 4;  // buffers of a device that wait for the next call

struct bounce_buf {
  char* p = nullptr;
  hipEvent_t done[BOUNCE_PIECES] = {};
};
static idle_by_device<bounce_buf>& bounces() {  // (the events belong to a device)
  static auto* b = new idle_by_device<bounce_buf>();
  return *b;
}
static void bounce_free(bounce_buf& b) {
  if (b.p) (void)hipHostFree(b.p);
  for (hipEvent_t e : b.done)
    if (e) (void)hipEventDestroy(e);
  b = bounce_buf();
}
static bool bounce_take(int dev, bounce_buf* b) {
  if (bounces().take(dev, b)) return true;
  bool ok = hipHostMalloc((void**)&b->p, 2 * BOUNCE_HALF, hipHostMallocDefault) == hipSuccess;
  for (hipEvent_t& e : b->done) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
  if (ok) return true;
  (void)hipGetLastError();
  bounce_free(*b);
  return false;
}
static void bounce_give(int dev, bounce_buf& b) {
  if (!bounces().give(dev, b, BOUNCE_KEPT)) bounce_free(b);
}
static_assert(pinned_buf::BYTES == 2 * BOUNCE_HALF, "one kind of buffer");
void pinned_buf::take() {
  bounce_buf b;
  if (p_ || hipGetDevice(&dev_) != hipSuccess || !bounce_take(dev_, &b)) return;
  p_ = b.p;
  std::copy(b.done, b.done + EVENTS, done_);
}
void pinned_buf::give() {
  if (!p_) return;
  bounce_buf b;
  b.p = p_;
  std::copy(done_, done_ + EVENTS, b.done);
  bounce_give(dev_, b);
  p_ = nullptr;
}
static void bounce_trim() { bounces().drain(bounce_free); }

__global__ void __launch_bounds__(256) k_copy_words(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, int n) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) dst[i] = src[i];
}

// Upwards: all arrays as one run of pieces of a quarter of a buffer, the next on its way into the buffer while others go over
// the link.  A matrix from 2 arrays of 2.4 MB: 210 us, 270 array by array in halves of a buffer.
static hipError_t bounce_up(const copy_part* parts, int n_parts) {
  constexpr size_t PIECE = 2 * BOUNCE_HALF / BOUNCE_PIECES;
  bounce_buf B;
  int dev = 0;
  hipError_t e = hipSuccess;
  if (hipGetDevice(&dev) != hipSuccess || !bounce_take(dev, &B)) {
    for (int q = 0; q < n_parts && e == hipSuccess; q++) e = hipMemcpy(parts[q].dst, parts[q].src, parts[q].bytes, hipMemcpyHostToDevice);
    return e;
  }
  hipStream_t st = stream();
  int k = 0;
  for (int q = 0; q < n_parts && e == hipSuccess; q++)
    for (size_t off = 0; off < parts[q].bytes && e == hipSuccess; off += PIECE, k++) {
      const int b = k % BOUNCE_PIECES;
      char* buf = B.p + b * PIECE;
      char* dst = (char*)parts[q].dst + off;
      const size_t n = parts[q].bytes - off < PIECE ? parts[q].bytes - off : PIECE;
      if (k >= BOUNCE_PIECES) e = hipEventSynchronize(B.done[b]);
      if (e != hipSuccess) break;
      memcpy(buf, (const char*)parts[q].src + off, n);
      if (n <= BOUNCE_KERNEL && n % 4 == 0 && (uintptr_t)dst % 4 == 0) {
        hipLaunchKernelGGL(k_copy_words, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, st, (const uint32_t*)buf, (uint32_t*)dst, (int)(n / 4));
        e = hipGetLastError();
      } else {
        e = piece_copy(dst, buf, n, hipMemcpyHostToDevice, st);
      }
      if (e == hipSuccess) e = hipEventRecord(B.done[b], st);
    }
  const hipError_t es = hipStreamSynchronize(st);
  bounce_give(dev, B);
  return e == hipSuccess ? es : e;
}

static hipError_t bounce_down(char* dst, const char* src, size_t bytes) {
  bounce_buf B;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || !bounce_take(dev, &B)) return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
  hipStream_t st = stream();
  hipError_t e = hipSuccess;
  if (bytes <= BOUNCE_KERNEL && bytes % 4 == 0 && (uintptr_t)src % 4 == 0) {
    const int n = (int)(bytes / 4);
    hipLaunchKernelGGL(k_copy_words, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (const uint32_t*)src,
                       (uint32_t*)B.p, n);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e == hipSuccess) memcpy(dst, B.p, bytes);
  } else if (bytes <= 2 * BOUNCE_HALF) {
    // both halves under way at once
    const size_t n0 = bytes < BOUNCE_HALF / 2 ? bytes : bytes / 2 / 16 * 16;
    e = piece_copy(B.p, src, n0, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipEventRecord(B.done[0], st);
    if (e == hipSuccess && n0 < bytes) e = piece_copy(B.p + n0, src + n0, bytes - n0, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) fetch_pages(dst, bytes);
    if (e == hipSuccess) e = hipEventSynchronize(B.done[0]);
    if (e == hipSuccess) memcpy(dst, B.p, n0);
    const hipError_t es = hipStreamSynchronize(st);
    if (e == hipSuccess) e = es;
    if (e == hipSuccess && n0 < bytes) memcpy(dst + n0, B.p + n0, bytes - n0);
  } else {
    size_t at[2] = {0, 0}, len[2] = {0, 0};
    int k = 0;
    for (size_t off = 0; off < bytes && e == hipSuccess; off += BOUNCE_HALF, k++) {
      const int b = k & 1;
      char* buf = B.p + b * BOUNCE_HALF;
      const size_t n = bytes - off < BOUNCE_HALF ? bytes - off : BOUNCE_HALF;
      if (k >= 2) e = hipEventSynchronize(B.done[b]);
      if (e != hipSuccess) break;
      if (len[b]) memcpy(dst + at[b], buf, len[b]);
      e = piece_copy(buf, src + off, n, hipMemcpyDeviceToHost, st);
      at[b] = off;
      len[b] = n;
      if (e == hipSuccess) e = hipEventRecord(B.done[b], st);
      if (e == hipSuccess) fetch_pages(dst + off, n);
    }
    const hipError_t es = hipStreamSynchronize(st);
    if (e == hipSuccess) e = es;
    if (e == hipSuccess)
      for (int i = k >= 2 ? k - 2 : 0; i < k; i++) memcpy(dst + at[i & 1], B.p + (i & 1) * BOUNCE_HALF, len[i & 1]);
  }
  if (e != hipSuccess) (void)hipStreamSynchronize(st);  // (nothing may still be on its way to the buffer)
  bounce_give(dev, B);
  return e;
}

constexpr int GATHER_PARTS = 4;
struct gather_parts {
  const uint32_t* src[GATHER_PARTS];
  int words[GATHER_PARTS], at[GATHER_PARTS];  // `at`: a multiple of four words
};
// Part blockIdx.y to dst, in 16-byte pieces where it is aligned (the rest of a part: single words).
__global__ void __launch_bounds__(256) k_gather_parts(gather_parts p, uint32_t* __restrict__ dst) {
  const uint32_t* src = p.src[blockIdx.y];
  uint32_t* to = dst + p.at[blockIdx.y];
  const int n = p.words[blockIdx.y], quads = ((uintptr_t)src & 15) == 0 ? n / 4 : 0;
  for (int i = blockIdx.x * 1024 + threadIdx.x; i < quads; i += gridDim.x * 1024) {
    uint4 v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) v[u] = reinterpret_cast<const uint4*>(src)[i + 256 * u < quads ? i + 256 * u : i];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (i + 256 * u < quads) reinterpret_cast<uint4*>(to)[i + 256 * u] = v[u];
  }
  for (int i = 4 * quads + blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) to[i] = src[i];
}

hipError_t gather_queue(const copy_part* parts, int n_parts, char* buf) {
  size_t at = 0;
  hipError_t e = hipSuccess;
  for (int q = 0; q < n_parts && e == hipSuccess; q += GATHER_PARTS) {
    gather_parts g = {};
    size_t most = 0;
    for (int i = 0; i < GATHER_PARTS && q + i < n_parts; i++) {
      const copy_part& p = parts[q + i];
      g.src[i] = (const uint32_t*)p.src;
      g.words[i] = (int)(p.bytes / 4);
      g.at[i] = (int)(at / 4);
      at += gather_room(p.bytes);
      most = most > p.bytes ? most : p.bytes;
    }
    const int wgs = (int)((most + 16383) / 16384);
    hipLaunchKernelGGL(k_gather_parts, dim3(wgs < COPY_WGS ? wgs : COPY_WGS, GATHER_PARTS), dim3(256), 0, stream(), g, (uint32_t*)buf);
    e = hipGetLastError();
  }
  return e;
}
void gather_take(const copy_part* parts, int n_parts, const char* buf) {
  for (int q = 0; q < n_parts; buf += gather_room(parts[q].bytes), q++) memcpy(parts[q].dst, buf, parts[q].bytes);
}

// Several short arrays down as one: a kernel writes them to a bounce buffer side by side, one wait for all.
// (Two arrays of 240 KB: one wait and 10 us of writes where the engine's copies took two waits and 14 us each before
// they began.)
static hipError_t gather_down(const copy_part* parts, int n_parts) {
  pinned_buf B;
  B.take();
  hipError_t e = hipSuccess;
  if (!B.p()) {
    for (int q = 0; q < n_parts && e == hipSuccess; q++) e = hipMemcpy(parts[q].dst, parts[q].src, parts[q].bytes, hipMemcpyDeviceToHost);
    return e;
  }
  e = gather_queue(parts, n_parts, B.p());
  if (e == hipSuccess)
    for (int q = 0; q < n_parts; q++) fetch_pages(parts[q].dst, parts[q].bytes);
  const hipError_t es = hipStreamSynchronize(stream());
  if (e == hipSuccess) e = es;
  if (e == hipSuccess) gather_take(parts, n_parts, B.p());
  return e;
}

// Short parts through bounce buffers (downwards as many at once as one holds), the rest in one run of pieces.
template <bool UP>
static hipError_t copy_parts(const copy_part* parts, int n_parts) {
  std::vector<copy_part> large, few;
  size_t held = 0;
  hipError_t e = hipSuccess;
  auto flush = [&]() {
    if (UP && !few.empty()) e = bounce_up(few.data(), (int)few.size());
    else if (few.size() > 1) e = gather_down(few.data(), (int)few.size());
    else if (few.size() == 1) e = bounce_down((char*)few[0].dst, (const char*)few[0].src, few[0].bytes);
    few.clear();
    held = 0;
    return e;
  };
  for (int i = 0; i < n_parts; i++) {
    const copy_part& q = parts[i];
    if (q.bytes >= STAGED_MIN) {
      large.push_back(q);
    } else if (UP) {
      if (q.bytes) few.push_back(q);
    } else if (q.bytes && q.bytes + 16 <= 2 * BOUNCE_HALF && q.bytes % 4 == 0 && (uintptr_t)q.src % 4 == 0) {
      if (held + q.bytes + 16 > 2 * BOUNCE_HALF && flush() != hipSuccess) return e;
      few.push_back(q);
      held += q.bytes + 16;
    } else if (q.bytes) {
      e = bounce_down((char*)q.dst, (const char*)q.src, q.bytes);
      if (e != hipSuccess) return e;
    }
  }
  if (flush() != hipSuccess) return e;
  return large.empty() ? hipSuccess : staged_copy<UP>(large.data(), (int)large.size());
}

hipError_t copy_up_parts(std::initializer_list<copy_part> parts) { return copy_parts<true>(parts.begin(), (int)parts.size()); }
hipError_t copy_down_parts(const copy_part* parts, int n_parts) { return copy_parts<false>(parts, n_parts); }
hipError_t copy_up(void* dst_dev, const void* src_host, size_t bytes) {
  const copy_part q{dst_dev, src_host, bytes};
  return copy_parts<true>(&q, 1);
}
hipError_t copy_down(void* dst_host, const void* src_dev, size_t bytes) {
  const copy_part q{dst_host, src_dev, bytes};
  return copy_parts<false>(&q, 1);
}

// A few pinned words that kernels write results into (one stream synchronisation then replaces a
// device-to-host copy of some bytes and its round trip); one set per host thread.
int host_words(unsigned long long** out) {
  static thread_local unsigned long long* words = nullptr;
  if (!words) {
    DN_HIP(hipHostMalloc((void**)&words, (2 * HOST_WORDS + HOST_STAMPS) * sizeof(unsigned long long), hipHostMallocDefault));
  }
  *out = words;
  return 0;
}
int host_waited_words(unsigned long long** out) {
  DN_TRY(host_words(out));
  *out += HOST_WORDS;
  return 0;
}
hipError_t wait_words(const unsigned long long* words, int n, hipStream_t st) {
  const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
  int i = 0;
  auto here = [&] {
    while (i < n && __atomic_load_n(words + i, __ATOMIC_ACQUIRE) != WORD_NONE) i++;
    return i == n;
  };
  while (!here() && std::chrono::steady_clock::now() < until) {
  }
  if (i == n) return hipSuccess;
  const hipError_t e = hipStreamSynchronize(st);
  return e != hipSuccess || here() ? e : hipErrorUnknown;
}
int host_stamps(unsigned long long** out) {
  DN_TRY(host_words(out));
  *out += 2 * HOST_WORDS;
  return 0;
}

}  // namespace dn

using namespace dn;

DN_API int dnpeff_release_cached(void) {
  clear_error();
  DN_HIP(hipStreamSynchronize(stream()));
  pool_trim();
  stage_trim();
  bounce_trim();
  return 0;
}
