// Staged host <-> device copies (see hostcopy.hpp).
#include "hostcopy.hpp"

#include "common.hpp"
#include "copypool.hpp"

#include <algorithm>
#include <atomic>
#include <mutex>

namespace cdn {
namespace {

// One pinned region, cut into 4 buffers of 16 MB, or 2 of 32 MB for copies of
// 512 MB and more.  A chunk is a quarter of the copy (1 to 16 MB), so that
// short copies overlap their DMA with the host threads too and the last
// chunk's host copy, which nothing overlaps, is short.  Measured with fresh
// destination pages, GB/s (2 buffers of 32 MB, everything below 16 MB through
// the runtime -> this): to the host 6.5 MB 7.2 -> 14, 12 MB 10 -> 19, 67 MB
// 29 -> 39, 134 MB 37 -> 43, 311 MB 41 -> 46; to the device 24 MB 34 -> 42,
// 67 MB 41 -> 47.  At 1 GB 32 MB chunks stay ahead (49.6 and 54.4 against
// 48.8 and 53.4 of 16 MB).
constexpr size_t kPinned = 64UL << 20;
constexpr size_t kMinChunk = 1UL << 20;
constexpr int kMaxBufs = 4;
// smaller copies go straight through the runtime: its pageable uploads reach
// 33 GB/s from 4 MB on, its downloads 4 to 11
constexpr size_t kDirectUp = 16UL << 20, kDirectDown = 2UL << 20;
// a stream made for the call takes 50 us more for its first copies into pinned
// memory: affine and deskew, ms through the runtime and staged: 2.1 MB 0.367 and
// 0.420, 3 MB 0.43 and 0.465, 3.9 MB 0.505 and 0.515, 4.9 MB 0.58 and 0.54
constexpr size_t kDirectFresh = 9UL << 19;
// Downloads below this size keep out of each other's way: they hold the buffers
// for the copy alone, not while their stream's kernels run, at most two wait for
// one of them, and any more, or any beside a larger copy, go through the runtime.
// Threads that fetch results side by side, ms per round: all through the runtime,
// each in turn through the buffers, this: 8 of 4.2 MB 0.82, 1.45, 0.83; 8 of
// 12.6 MB 2.42, 2.71, 2.42; 4 of 12.6 MB 1.22, 1.34, 1.22; with 10 iterations
// before each, 4 of 12.6 MB 3.78, 2.86, 2.87; 8 of them 5.31, 5.54, 5.33.  (One
// waiting instead of two: 3.11 and 5.21.)
constexpr size_t kShared = 16UL << 20;

struct Chunks {
  size_t cap, chunk, n;  // bytes per buffer, bytes per chunk, chunks
  int bufs;
  explicit Chunks(size_t bytes) {
    const bool large = bytes >= (512UL << 20);
    cap = large ? 32UL << 20 : 16UL << 20;
    bufs = (int)(kPinned / cap);
    chunk = large ? cap : std::min(cap, (bytes / 4 + kMinChunk - 1) / kMinChunk * kMinChunk);
    n = (bytes + chunk - 1) / chunk;
  }
  size_t buf(size_t i) const { return i % (size_t)bufs; }
  size_t off(size_t i) const { return i * chunk; }
  size_t len(size_t i, size_t bytes) const { return std::min(chunk, bytes - off(i)); }
};

constexpr int kWaiting = 2, kLarge = kWaiting + 1;

struct Stage {
  std::mutex mu;
  std::atomic<int> users{0};  // holding or waiting: a copy below kShared counts 1, any other kLarge
  CopyPool* pool = nullptr;
  void* base = nullptr;  // pinned, portable across devices
  char* at(const Chunks& c, size_t i) const { return static_cast<char*>(base) + c.buf(i) * c.cap; }
  void ensure() {
    if (!base) CDN_HIP(hipHostMalloc(&base, kPinned, hipHostMallocPortable));
    if (!pool) pool = new CopyPool;
  }
};

// The events of one call (the last DMA through each buffer), created on the
// device of the call's stream and destroyed when the call returns, after every
// DMA through the staging buffers has finished.  No
// event outlives its call, so none is ever waited on after the stream it
// was recorded on has been destroyed (the caller may destroy it right after
// the call).
struct CallEvents {
  hipEvent_t e[kMaxBufs] = {};
  explicit CallEvents(hipStream_t st) {
    int dev = 0, cur = 0;
    CDN_HIP(hipStreamGetDevice(st, &dev));
    CDN_HIP(hipGetDevice(&cur));
    if (cur != dev) CDN_HIP(hipSetDevice(dev));
    hipError_t rc = hipSuccess;
    for (int i = 0; i < kMaxBufs && rc == hipSuccess; ++i) rc = hipEventCreateWithFlags(&e[i], hipEventDisableTiming);
    if (cur != dev) (void)hipSetDevice(cur);
    if (rc != hipSuccess) {
      release();
      CDN_HIP(rc);
    }
  }
  void release() {
    for (hipEvent_t& x : e)
      if (x) {
        (void)hipEventDestroy(x);
        x = nullptr;
      }
  }
  ~CallEvents() { release(); }
};

struct Use {
  Stage& s;
  const int n;
  const int before;
  Use(Stage& st, int k) : s(st), n(k), before(st.users.fetch_add(k)) {}
  ~Use() { s.users.fetch_sub(n); }
};

// process lifetime: the pinned buffers are released when the process ends
Stage& stage() {
  static Stage* s = new Stage;
  return *s;
}

// on a failed call: no DMA through the staging buffers may still be in
// flight when the next call takes them (the error itself is reported)
void drain(hipStream_t st) { (void)hipStreamSynchronize(st); }

}  // namespace

void copy_to_device(hipStream_t st, void* dev, const void* host, size_t bytes) {
  if (bytes < kDirectUp) {
    CDN_HIP(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st));
    return;
  }
  Stage& S = stage();
  const Use use(S, kLarge);
  std::lock_guard<std::mutex> lock(S.mu);
  S.ensure();
  CallEvents E(st);
  const Chunks c(bytes);
  try {
    for (size_t i = 0; i < c.n; ++i) {
      hipEvent_t ev = E.e[c.buf(i)];
      if (i >= (size_t)c.bufs) CDN_HIP(hipEventSynchronize(ev));  // the DMA that used this buffer before
      S.pool->copy(S.at(c, i), static_cast<const char*>(host) + c.off(i), c.len(i, bytes));
      CDN_HIP(hipMemcpyAsync(static_cast<char*>(dev) + c.off(i), S.at(c, i), c.len(i, bytes), hipMemcpyHostToDevice,
                             st));
      CDN_HIP(hipEventRecord(ev, st));
    }
    // the staging buffers are free for the next call (one stream: the last
    // DMA ends after all before it)
    CDN_HIP(hipEventSynchronize(E.e[c.buf(c.n - 1)]));
  } catch (...) {
    drain(st);
    throw;
  }
}

void copy_to_host(hipStream_t st, void* host, const void* dev, size_t bytes, bool fresh_stream) {
  if (bytes < (fresh_stream ? kDirectFresh : kDirectDown)) {
    CDN_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st));
    CDN_HIP(hipStreamSynchronize(st));
    return;
  }
  Stage& S = stage();
  if (bytes < kShared && hipStreamQuery(st) != hipSuccess) {  // (a synchronisation of an idle stream takes 25 us)
    if (hipPeekAtLastError() == hipErrorNotReady) (void)hipGetLastError();  // the answer, no error of a later launch
    CDN_HIP(hipStreamSynchronize(st));
  }
  const Use use(S, bytes < kShared ? 1 : kLarge);
  if (bytes < kShared && use.before > kWaiting) {
    CDN_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st));
    CDN_HIP(hipStreamSynchronize(st));
    return;
  }
  std::lock_guard<std::mutex> lock(S.mu);
  S.ensure();
  CallEvents E(st);
  const Chunks c(bytes);
  auto issue = [&](size_t i) {
    CDN_HIP(hipMemcpyAsync(S.at(c, i), static_cast<const char*>(dev) + c.off(i), c.len(i, bytes),
                           hipMemcpyDeviceToHost, st));
    CDN_HIP(hipEventRecord(E.e[c.buf(i)], st));
  };
  try {
    size_t issued = 0;
    for (size_t i = 0; i < c.n; ++i) {
      // the buffer of chunk j was emptied by the host copy of chunk j - bufs < i
      for (; issued < c.n && issued < i + (size_t)c.bufs; ++issued) issue(issued);
      CDN_HIP(hipEventSynchronize(E.e[c.buf(i)]));
      S.pool->copy(static_cast<char*>(host) + c.off(i), S.at(c, i), c.len(i, bytes));
    }
  } catch (...) {
    drain(st);
    throw;
  }
}

}  // namespace cdn
