// Copies between pageable host arrays (Java arrays handed over by JNA, numpy
// arrays) and device memory for the entry points whose contract is host
// arrays.  Large copies go through two pinned staging buffers per device: the
// DMA engine moves one chunk while host threads copy another between a staging
// buffer and the pageable array, so the single-threaded pageable copy of the
// runtime is not the bound.  Small copies use the runtime directly.  Each call
// returns when its copy is done.  The two 16 MiB pinned buffers of a device are
// allocated at its first large copy and held until the process ends; large
// copies on one device are serialised by a mutex (the JNA hooks are called from
// one thread per device).  The all-or-nothing variant keeps one more pinned
// buffer per device, as large as the largest such copy so far, also held until
// the process ends.
//
// Downloads are bound by the host: the pages of a new array are first touched
// here.  Their threads are started once per call and take pieces of 8 MiB chunks
// (halves of the buffers).  A 67 MB result into a new array: eight threads started
// for each 16 MiB chunk 2.4 ms; 14 threads and three halves 1.9, four halves 2.0,
// two 2.3, eight threads 2.0, pieces of 512 KiB 2.0 to 2.5.  Uploads gain nothing
// from it (67 MB both ways 3.57 and 3.67 ms) and keep whole buffers, cut once
// per chunk.
#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "mvd_internal.h"

namespace mvd {
namespace {

constexpr size_t kStageChunk = 16u << 20;  // bytes per staging buffer
constexpr size_t kHalf = kStageChunk / 2;  // a download's chunk
constexpr int kHalves = 3;                 // in flight
constexpr size_t kStageMin = 8u << 20;     // smaller copies use the runtime
constexpr size_t kPiece = 1u << 20;        // bytes a thread copies at a time
constexpr int kMaxDevices = 64;
constexpr int kTeam = 14;  // threads of a download, beside the caller's

struct Stage {
  std::mutex mu;
  void* buf[2] = {nullptr, nullptr};
  hipEvent_t ev[kHalves] = {};
  bool ready = false;
  void* whole = nullptr;  // pinned buffer of the all-or-nothing copies (grows, held)
  size_t whole_cap = 0;
  char* half(int i) { return static_cast<char*>(buf[i / 2]) + (i % 2) * kHalf; }
};
Stage g_stage[kMaxDevices];

int copy_threads() {
  static const int n = [] {
    const unsigned hw = std::thread::hardware_concurrency();
    return (int)std::max(1u, std::min(8u, hw ? hw / 2 : 1u));
  }();
  return n;
}

// memcpy split over a few threads (the calling thread takes the first part)
void parallel_copy(void* dst, const void* src, size_t bytes) {
  const int t = bytes >= (2u << 20) ? copy_threads() : 1;
  if (t <= 1) {
    std::memcpy(dst, src, bytes);
    return;
  }
  const size_t part = (bytes / t + 63) & ~size_t(63);
  std::vector<std::thread> th;
  th.reserve(t - 1);
  for (int i = 1; i < t; ++i) {
    const size_t off = part * i;
    if (off >= bytes) break;
    const size_t n = std::min(part, bytes - off);
    auto copy = [=] { std::memcpy(static_cast<char*>(dst) + off, static_cast<const char*>(src) + off, n); };
    try {
      th.emplace_back(copy);
    } catch (const std::system_error&) {  // no thread to be had
      copy();
    }
  }
  std::memcpy(dst, src, std::min(part, bytes));
  for (auto& x : th) x.join();
}

// Host threads of one download: chunks are posted in order and copied in pieces; the
// posting thread takes pieces too while it waits for a chunk.  At most kHalves
// chunks are unfinished at a time.  With no thread to be had the posting thread
// copies everything.
class CopyTeam {
 public:
  explicit CopyTeam(size_t bytes) {
    const unsigned hw = std::thread::hardware_concurrency();
    const int want = (int)std::min<size_t>({kTeam, hw ? hw / 2 : 1, bytes / (1u << 20)});
    try {
      for (; n_ < want; ++n_) th_[n_] = std::thread([this] { work(); });
    } catch (const std::system_error&) {
    }
  }
  ~CopyTeam() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    more_.notify_all();
    for (int i = 0; i < n_; ++i) th_[i].join();
  }
  // chunk number `k` (0, 1, 2, ...)
  void post(int k, void* dst, const void* src, size_t bytes) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      jobs_[k % kHalves] = {static_cast<char*>(dst), static_cast<const char*>(src), bytes, 0, 0};
      posted_ = k + 1;
    }
    more_.notify_all();
  }
  void wait(int k) {
    std::unique_lock<std::mutex> lk(mu_);
    Job& j = jobs_[k % kHalves];
    while (j.done < j.bytes)
      if (!take(lk)) done_.wait(lk);
  }

 private:
  struct Job {
    char* dst = nullptr;
    const char* src = nullptr;
    size_t bytes = 0, next = 0, done = 0;
  };
  // copies one piece of the first chunk that has one left (mu_ is released meanwhile)
  bool take(std::unique_lock<std::mutex>& lk) {
    for (; first_ < posted_; ++first_) {
      Job& j = jobs_[first_ % kHalves];
      if (j.next >= j.bytes) continue;
      const size_t at = j.next, n = std::min(kPiece, j.bytes - at);
      j.next += n;
      lk.unlock();
      std::memcpy(j.dst + at, j.src + at, n);
      lk.lock();
      j.done += n;
      if (j.done >= j.bytes) done_.notify_all();
      return true;
    }
    return false;
  }
  void work() {
    std::unique_lock<std::mutex> lk(mu_);
    while (!stop_)
      if (!take(lk)) more_.wait(lk);
  }

  std::mutex mu_;
  std::condition_variable more_, done_;
  Job jobs_[kHalves];
  int posted_ = 0, first_ = 0;  // chunks posted; first chunk that may have pieces left
  bool stop_ = false;
  std::thread th_[kTeam];
  int n_ = 0;
};

hipError_t stage_for(int dev, Stage** out) {
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  Stage& s = g_stage[dev];
  if (!s.ready) {
    for (auto& b : s.buf) {
      const hipError_t e = b ? hipSuccess : hipHostMalloc(&b, kStageChunk, hipHostMallocDefault);
      if (e != hipSuccess) return e;
    }
    for (auto& ev : s.ev) {
      const hipError_t e = ev ? hipSuccess : hipEventCreateWithFlags(&ev, hipEventDisableTiming);
      if (e != hipSuccess) return e;
    }
    s.ready = true;
  }
  *out = &s;
  return hipSuccess;
}

}  // namespace

hipError_t staged_h2d(void* dst, const void* src, size_t bytes, hipStream_t stream) {
  if (bytes < kStageMin) {
    hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  }
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lk(g_stage[std::clamp(dev, 0, kMaxDevices - 1)].mu);
  Stage* s = nullptr;
  if ((e = stage_for(dev, &s)) != hipSuccess) return e;
  size_t done = 0;
  for (int k = 0; done < bytes && e == hipSuccess; ++k) {
    const int b = k & 1;
    const size_t n = std::min(kStageChunk, bytes - done);
    if (k >= 2) e = hipEventSynchronize(s->ev[b]);  // its previous DMA has read the buffer
    if (e != hipSuccess) break;
    parallel_copy(s->buf[b], static_cast<const char*>(src) + done, n);
    e = hipMemcpyAsync(static_cast<char*>(dst) + done, s->buf[b], n, hipMemcpyHostToDevice, stream);
    if (e == hipSuccess) e = hipEventRecord(s->ev[b], stream);
    done += n;
  }
  const hipError_t es = hipStreamSynchronize(stream);
  return e != hipSuccess ? e : es;
}

hipError_t staged_d2h(void* dst, const void* src, size_t bytes, hipStream_t stream) {
  if (bytes < kStageMin) {
    hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  }
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lk(g_stage[std::clamp(dev, 0, kMaxDevices - 1)].mu);
  Stage* s = nullptr;
  if ((e = stage_for(dev, &s)) != hipSuccess) return e;
  {
    CopyTeam team(bytes);
    const int chunks = (int)((bytes + kHalf - 1) / kHalf);
    auto size = [&](int k) { return std::min(kHalf, bytes - k * kHalf); };
    auto dma = [&](int k) {
      const int b = k % kHalves;
      const hipError_t r = hipMemcpyAsync(s->half(b), static_cast<const char*>(src) + k * kHalf, size(k),
                                          hipMemcpyDeviceToHost, stream);
      return r == hipSuccess ? hipEventRecord(s->ev[b], stream) : r;
    };
    int copied = 0;  // chunks posted
    for (int k = 0; k < std::min(chunks, kHalves) && e == hipSuccess; ++k) e = dma(k);
    for (int k = 0; k < chunks && e == hipSuccess; ++k) {
      const int b = k % kHalves;
      if ((e = hipEventSynchronize(s->ev[b])) != hipSuccess) break;
      team.post(k, static_cast<char*>(dst) + k * kHalf, s->half(b), size(k));
      copied = k + 1;
      // the buffer of the chunk before is the next to be filled again
      if (k >= 1 && k - 1 + kHalves < chunks) {
        team.wait(k - 1);
        e = dma(k - 1 + kHalves);
      }
    }
    for (int k = std::max(0, copied - kHalves); k < copied; ++k) team.wait(k);
  }
  const hipError_t es = hipStreamSynchronize(stream);
  return e != hipSuccess ? e : es;
}

// Device to host where the host array must stay as it was unless the whole
// copy succeeds: the DMA fills one pinned buffer of the full size, and only
// after it has completed without error is the host array overwritten.
hipError_t staged_d2h_all_or_nothing(void* dst, const void* src, size_t bytes, hipStream_t stream) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  Stage& s = g_stage[dev];
  std::lock_guard<std::mutex> lk(s.mu);
  if (s.whole_cap < bytes) {
    if (s.whole) (void)hipHostFree(s.whole);
    s.whole = nullptr;
    s.whole_cap = 0;
    if ((e = hipHostMalloc(&s.whole, bytes, hipHostMallocDefault)) != hipSuccess) return e;
    s.whole_cap = bytes;
  }
  if ((e = hipMemcpyAsync(s.whole, src, bytes, hipMemcpyDeviceToHost, stream)) != hipSuccess) return e;
  if ((e = hipStreamSynchronize(stream)) != hipSuccess) return e;
  parallel_copy(dst, s.whole, bytes);
  return hipSuccess;
}

}  // namespace mvd
