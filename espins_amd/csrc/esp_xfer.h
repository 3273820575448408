// esp_xfer.h -- results from the device to the caller's (pageable) memory, shared by the
// single-context and the batched engine.
//
// A copy into pageable memory goes through the runtime's own staging, one chunk after the other,
// at about 10 GB/s with the page faults of a fresh destination on top (FCC 32^3 x 64: 201 MB of
// spins, 20 ms), and every small copy waits for the stream by itself.  Here
//  * spins go in chunks of kXChunk through pinned slots, one per worker thread: while one thread's
//    chunk is turned into reference order and copied by the GPU, the others move theirs into the
//    destination (and take its page faults);
//  * small results of one call are copied into one pinned page and waited for once.
// Pinned memory takes milliseconds to allocate and to free, longer than a small run, so a context
// or batch that finds no buffers waiting allocates them only after kXFirst bytes of spins or
// kXAsks small reads; until then it copies as it comes.  It gives its buffers back when it is
// destroyed; up to kXKeep sets wait for the next one, and the last context or batch to go frees
// them all.  Workers live for one call.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace espx {

constexpr size_t kXChunk = size_t(3) << 20;      // bytes per slot (a multiple of 24)
constexpr int kXSlots = 8;
constexpr size_t kXSmall = size_t(1) << 18;
constexpr size_t kXFirst = size_t(64) << 20;
constexpr int kXAsks = 32;

struct Xfer {
  int device = -1;
  char *pin = nullptr, *dev = nullptr, *small = nullptr;
  hipEvent_t ev[kXSlots] = {};
  int slots = 0;                                 // slots allocated
  size_t seen = 0;                               // bytes of spins read so far
  int asks = 0;                                  // small reads so far

  void release() {
    for (auto &e : ev)
      if (e) (void)hipEventDestroy(e);
    if (pin) (void)hipHostFree(pin);
    if (dev) (void)hipFree(dev);
    if (small) (void)hipHostFree(small);
    *this = Xfer{};
  }

  // At least n slots; buffers only grow.  Without pinned memory (pin stays null) the chunks are
  // copied straight into the destination.
  hipError_t reserve(int n) {
    if (n <= slots) return hipSuccess;
    if (pin) (void)hipHostFree(pin);
    if (dev) (void)hipFree(dev);
    pin = dev = nullptr;
    slots = 0;
    if (hipHostMalloc((void **)&pin, n * kXChunk, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      pin = nullptr;
    }
    hipError_t e = hipMalloc((void **)&dev, n * kXChunk);
    for (int i = 0; i < n && e == hipSuccess; ++i)
      if (!ev[i]) e = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
    if (e == hipSuccess) slots = n;
    return e;
  }
};

constexpr size_t kXKeep = 4;
struct XferPool {
  std::mutex mu;
  std::vector<Xfer> idle;
  int users = 0;
};
inline XferPool &xfer_pool() {
  static XferPool *p = [] {                // never destroyed: contexts may outlive static objects
    auto *q = new XferPool();
    q->idle.reserve(kXKeep);
    return q;
  }();
  return *p;
}
// A context or batch on `device` begins / ends.
inline void xfer_open(Xfer &x, int device) {
  XferPool &p = xfer_pool();
  std::lock_guard<std::mutex> lk(p.mu);
  ++p.users;
  x.device = device;
}
inline void xfer_take(Xfer &x) {           // buffers of an earlier owner, if any wait
  if (x.dev || x.small) return;
  XferPool &p = xfer_pool();
  std::lock_guard<std::mutex> lk(p.mu);
  for (size_t i = 0; i < p.idle.size(); ++i)
    if (p.idle[i].device == x.device) {
      x = p.idle[i];       // (its counts, too: they only grow)
      p.idle.erase(p.idle.begin() + i);
      return;
    }
}
inline void xfer_close(Xfer &x) {          // the owner's stream is idle
  XferPool &p = xfer_pool();
  std::lock_guard<std::mutex> lk(p.mu);
  if (x.device < 0) return;
  if (x.dev || x.small) {
    if (p.idle.size() < kXKeep && p.users > 1) p.idle.push_back(x);
    else x.release();
  }
  x = Xfer{};
  if (--p.users == 0) {
    for (auto &i : p.idle) i.release();
    p.idle.clear();
  }
}

// Spins of R replicas x N sites (reference order) into out.  src_rep: replica of each output row,
// or null.
template <class K>
hipError_t xfer_spins(K kernel, Xfer &x, int device, hipStream_t stream, const double *sp, const int *ref2dev,
                      const int *src_rep, int N, int Ns, int R, double *out) {
  const size_t total = (size_t)N * R, per = kXChunk / 24;      // spins
  const size_t chunks = (total + per - 1) / per;
  const int nt = (int)std::min<size_t>(chunks, kXSlots);
  xfer_take(x);
  x.seen += 24 * total;
  hipError_t e;
  if (!x.dev && x.seen < kXFirst) {
    double *d = nullptr;
    if ((e = hipMalloc((void **)&d, 24 * total)) != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, sp, ref2dev, src_rep, N,
                       Ns, (size_t)0, total, d);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(out, d, 24 * total, hipMemcpyDeviceToHost, stream);
    const hipError_t q = hipStreamSynchronize(stream);
    (void)hipFree(d);
    return e == hipSuccess ? q : e;
  }
  e = x.reserve(nt);
  if (e != hipSuccess) return e;
  std::atomic<int> err{hipSuccess};
  auto work = [&](int t) {
    hipError_t q = hipSetDevice(device);
    for (size_t c = t; c < chunks && q == hipSuccess && err.load() == hipSuccess; c += nt) {
      const size_t t0 = c * per, n = std::min(per, total - t0);
      double *d = reinterpret_cast<double *>(x.dev + t * kXChunk);
      hipLaunchKernelGGL(kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, sp, ref2dev, src_rep,
                         N, Ns, t0, n, d);
      q = hipGetLastError();
      void *to = x.pin ? (void *)(x.pin + t * kXChunk) : (void *)(out + 3 * t0);
      if (q == hipSuccess) q = hipMemcpyAsync(to, d, 24 * n, hipMemcpyDeviceToHost, stream);
      if (q == hipSuccess) q = hipEventRecord(x.ev[t], stream);
      if (q == hipSuccess) q = hipEventSynchronize(x.ev[t]);
      if (q == hipSuccess && x.pin) std::memcpy(out + 3 * t0, x.pin + t * kXChunk, 24 * n);
    }
    if (q != hipSuccess) err = q;
  };
  std::vector<std::thread> th;
  try {
    for (int t = 1; t < nt; ++t) th.emplace_back(work, t);
  } catch (...) {                                // no more threads: this one does their chunks
    for (int t = (int)th.size() + 1; t < nt; ++t) work(t);
  }
  work(0);
  for (auto &t : th) t.join();
  if (err.load() != hipSuccess) (void)hipStreamSynchronize(stream);   // nothing in flight into the slots
  return (hipError_t)err.load();
}

// Small results of one call: add() queues copies on the stream, finish() waits once and hands
// them over.  What does not fit the page, or finds none, is copied directly.
class SmallRead {
 public:
  SmallRead(Xfer &x, hipStream_t s) : x_(x), s_(s) {
    xfer_take(x_);
    if (!x_.small && ++x_.asks > kXAsks && hipHostMalloc((void **)&x_.small, kXSmall, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      x_.small = nullptr;
    }
  }
  void add(void *dst, const void *src, size_t bytes) {
    if (e_ != hipSuccess || !bytes) return;
    if (!x_.small || n_ == kMax || used_ + bytes > kXSmall) {
      e_ = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s_);
      return;
    }
    e_ = hipMemcpyAsync(x_.small + used_, src, bytes, hipMemcpyDeviceToHost, s_);
    todo_[n_++] = {dst, used_, bytes};
    used_ += (bytes + 15) / 16 * 16;
  }
  hipError_t finish() {
    const hipError_t q = hipStreamSynchronize(s_);
    if (e_ == hipSuccess) e_ = q;
    if (e_ == hipSuccess)
      for (int i = 0; i < n_; ++i) std::memcpy(todo_[i].dst, x_.small + todo_[i].off, todo_[i].bytes);
    return e_;
  }

 private:
  static constexpr int kMax = 8;
  struct Item { void *dst; size_t off, bytes; };
  Xfer &x_;
  hipStream_t s_;
  hipError_t e_ = hipSuccess;
  size_t used_ = 0;
  int n_ = 0;
  Item todo_[kMax];
};

}  // namespace espx
