// Copies between pageable host arrays (Java arrays handed over by JNA, numpy
// arrays) and device memory for the entry points whose contract is host
// arrays.  Large copies go through three pinned staging buffers per device: the
// DMA engine moves some chunks while host threads copy others between their
// staging buffers and the pageable array, so the single-threaded pageable copy
// of the runtime is not the bound.  Small copies use the runtime directly.
// Each call returns when its copy is done.  The pinned buffers of a device are
// allocated at its first large copy and held until the process ends; large
// copies on one device are serialised by a mutex (the JNA hooks are called from
// one thread per device).  The all-or-nothing variant keeps one more pinned
// buffer per device, as large as the largest such copy so far, also held until
// the process ends.
//
// The threads are started once per call, not per chunk (starting eight costs
// about as much as the DMA of four MiB).  Sizes and counts by measurement, a
// 67 MB result into a new array and a 67 MB block both ways: two 16 MiB buffers
// with eight threads started per chunk 2.4 and 3.7 ms; 8 MiB, three buffers, 14
// threads, pieces of 1 MiB 1.9 and 3.7; two buffers 2.3 and 3.7; four buffers of
// 16 MiB 2.0 and 4.1; pieces of 512 KiB 2.0 to 2.5 and 4.2 to 4.8.
#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>

#include "mvd_internal.h"

namespace mvd {
namespace {

constexpr size_t kStageChunk = 8u << 20;   // bytes per staging buffer
constexpr int kStageBufs = 3;
constexpr size_t kStageMin = 8u << 20;     // smaller copies use the runtime
constexpr size_t kPiece = 1u << 20;        // bytes a thread copies at a time
constexpr int kMaxDevices = 64;
// into new pages many threads, whose page faults overlap; else eight with the poster
constexpr int kMaxCopyThreads = 14, kFillThreads = 7;

struct Stage {
  std::mutex mu;
  void* buf[kStageBufs] = {};
  hipEvent_t ev[kStageBufs] = {};
  bool ready = false;
  void* whole = nullptr;  // pinned buffer of the all-or-nothing copies (grows, held)
  size_t whole_cap = 0;
};
Stage g_stage[kMaxDevices];

// Host threads of one copy: chunks are posted in order and copied in pieces; the
// posting thread takes pieces too while it waits for a chunk.  At most kStageBufs
// chunks are unfinished at a time.  With no thread to be had the posting thread
// copies everything.
class CopyTeam {
 public:
  CopyTeam(size_t bytes, int threads, size_t piece) : piece_(piece) {
    const unsigned hw = std::thread::hardware_concurrency();
    const int want = (int)std::min<size_t>({(size_t)threads, hw ? hw / 2 : 1, bytes / (1u << 20)});
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
      jobs_[k % kStageBufs] = {static_cast<char*>(dst), static_cast<const char*>(src), bytes, 0, 0};
      posted_ = k + 1;
    }
    more_.notify_all();
  }
  void wait(int k) {
    std::unique_lock<std::mutex> lk(mu_);
    Job& j = jobs_[k % kStageBufs];
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
      Job& j = jobs_[first_ % kStageBufs];
      if (j.next >= j.bytes) continue;
      const size_t at = j.next, n = std::min(piece_, j.bytes - at);
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

  const size_t piece_;
  std::mutex mu_;
  std::condition_variable more_, done_;
  Job jobs_[kStageBufs];
  int posted_ = 0, first_ = 0;  // chunks posted; first chunk that may have pieces left
  bool stop_ = false;
  std::thread th_[kMaxCopyThreads];
  int n_ = 0;
};

hipError_t stage_for(int dev, Stage** out) {
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  Stage& s = g_stage[dev];
  if (!s.ready) {
    for (int b = 0; b < kStageBufs; ++b) {
      hipError_t e = s.buf[b] ? hipSuccess : hipHostMalloc(&s.buf[b], kStageChunk, hipHostMallocDefault);
      if (e == hipSuccess && !s.ev[b]) e = hipEventCreateWithFlags(&s.ev[b], hipEventDisableTiming);
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
  {
    CopyTeam team(bytes, kFillThreads, kPiece);
    const int chunks = (int)((bytes + kStageChunk - 1) / kStageChunk);
    auto size = [&](int k) { return std::min(kStageChunk, bytes - k * kStageChunk); };
    int posted = 0;
    for (int k = 0; k < chunks && e == hipSuccess; ++k) {
      // fill up to two buffers ahead of the DMA of chunk k
      for (; posted < chunks && posted < k + kStageBufs - 1 && e == hipSuccess; ++posted) {
        const int b = posted % kStageBufs;
        if (posted >= kStageBufs) e = hipEventSynchronize(s->ev[b]);  // its previous DMA has read the buffer
        if (e == hipSuccess) team.post(posted, s->buf[b], static_cast<const char*>(src) + posted * kStageChunk, size(posted));
      }
      if (e != hipSuccess) break;
      team.wait(k);
      const int b = k % kStageBufs;
      e = hipMemcpyAsync(static_cast<char*>(dst) + k * kStageChunk, s->buf[b], size(k), hipMemcpyHostToDevice, stream);
      if (e == hipSuccess) e = hipEventRecord(s->ev[b], stream);
    }
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
    CopyTeam team(bytes, kMaxCopyThreads, kPiece);
    const int chunks = (int)((bytes + kStageChunk - 1) / kStageChunk);
    auto size = [&](int k) { return std::min(kStageChunk, bytes - k * kStageChunk); };
    auto dma = [&](int k) {
      const int b = k % kStageBufs;
      const hipError_t r = hipMemcpyAsync(s->buf[b], static_cast<const char*>(src) + k * kStageChunk, size(k),
                                          hipMemcpyDeviceToHost, stream);
      return r == hipSuccess ? hipEventRecord(s->ev[b], stream) : r;
    };
    int copied = 0;  // chunks posted
    for (int k = 0; k < std::min(chunks, kStageBufs) && e == hipSuccess; ++k) e = dma(k);
    for (int k = 0; k < chunks && e == hipSuccess; ++k) {
      const int b = k % kStageBufs;
      if ((e = hipEventSynchronize(s->ev[b])) != hipSuccess) break;
      team.post(k, static_cast<char*>(dst) + k * kStageChunk, s->buf[b], size(k));
      copied = k + 1;
      // the buffer of the chunk before is the next to be filled again
      if (k >= 1 && k - 1 + kStageBufs < chunks) {
        team.wait(k - 1);
        e = dma(k - 1 + kStageBufs);
      }
    }
    for (int k = std::max(0, copied - kStageBufs); k < copied; ++k) team.wait(k);
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
  CopyTeam team(bytes, kFillThreads, kPiece);
  team.post(0, dst, s.whole, bytes);
  team.wait(0);
  return hipSuccess;
}

}  // namespace mvd
