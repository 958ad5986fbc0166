// Large copies between a caller's pageable host arrays and device memory.
//
// hipMemcpyAsync moves pageable memory through a staging buffer of the runtime with one host thread.
// Here a few worker threads each copy chunks between the caller's array and two pinned chunks of
// their own while the copy engine moves the others; page faults of a new destination are taken by
// all of them at once.  84 MB (32^3 elements, N = 3): to the device 2.85 -> 1.96 ms, back into a new
// array 8.2 -> 2.7 ms; 164 MB 5.5 -> 3.7 and 15.6 -> 4.3 ms; 10.5 MB back 0.60 -> 0.40 ms.
// (Pinned copies run at 57 GB/s here.)  Chunks of 1 and 2 MiB: every copy costs about 35 us of
// its own, 84 MB up in 2.75 and 2.15 ms; 8 MiB loses on small transfers; 8 workers gain nothing.
//
// The workers and their pinned chunks (32 MiB per device) are shared by the device's contexts and
// given back when the last context that used them is destroyed.  Making and giving them back takes
// 1.3 ms (2.5-4.5 ms more the first time in a process), which a context of one upload and one
// download does not get back below some 20 MiB: created, uploaded, run for 2 steps, downloaded and
// destroyed with workers of its own against the plain copies, 4 MiB 3.4 against 1.6 ms, 10 MiB
// 5.0 / 4.3, 16 MiB 6.25 / 6.2, 24 MiB 8.5 / 9.0, 48 MiB 14 / 17, 164 MiB 58 / 71.  So a context
// has them made when its own transfers amount to BUILD_BYTES (HostTransfers) and uses those that
// another context has had made from its first transfer on.  One transfer uses them at a time; a
// transfer that finds them busy (or could not make them) takes the plain copy.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>

namespace fx {

class HostCopy {
 public:
  static constexpr int WORKERS = 4;
  static constexpr size_t CHUNK = (size_t)4 << 20;
  // below these the plain copy: to the device while the chunks occupy two workers at most (arrays
  // not in the host's caches, plain / staged: 4 MiB 0.18 / 0.25 ms, 8 MiB 0.33 / 0.36, 10 MiB 0.40 / 0.36,
  // 14 MiB 0.54 / 0.465, 20 MiB 0.77 / 0.65; one array sent again and again is as fast either way from 10
  // to 16 MiB), from it while one worker has all of it (4 MiB 0.25 / 0.25, 5 MiB 0.30 / 0.255, 8 MiB
  // 0.48 / 0.35).
  static constexpr size_t MIN_UP = (size_t)9 << 20, MIN_DOWN = (size_t)5 << 20;
  static constexpr size_t BUILD_BYTES = (size_t)64 << 20;

  // The device's workers; where there are none, made if `make` says so (null if that fails), else null.
  static std::shared_ptr<HostCopy> get(int dev, bool make) noexcept
  {
    constexpr int MAXDEV = 64;
    static std::mutex mu;
    static std::weak_ptr<HostCopy> live[MAXDEV];
    if (dev < 0 || dev >= MAXDEV) return nullptr;
    try {
      std::lock_guard<std::mutex> lk(mu);
      std::shared_ptr<HostCopy> p = live[dev].lock();
      if (!p && make) {
        p.reset(new HostCopy(dev));
        if (!p->start()) return nullptr;
        live[dev] = p;
      }
      return p;
    } catch (...) {
      return nullptr;
    }
  }

  ~HostCopy()
  {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    wake_.notify_all();
    for (std::thread &t : th_)
      if (t.joinable()) t.join();
    Relaxed relaxed;
    for (Slot &s : slot_) {
      if (s.ev) (void)hipEventDestroy(s.ev);
      if (s.p) (void)hipHostFree(s.p);
    }
  }

  // Copies bytes and waits for them on the stream; false: not taken (busy), nothing was done.
  bool copy(void *dst, const void *src, size_t bytes, bool to_device, hipStream_t stream, hipError_t *err) noexcept
  {
    std::unique_lock<std::mutex> job(job_, std::try_to_lock);
    if (!job.owns_lock()) return false;
    {
      std::lock_guard<std::mutex> lk(mu_);
      dst_ = static_cast<char *>(dst);
      src_ = static_cast<const char *>(src);
      bytes_ = bytes;
      to_device_ = to_device;
      stream_ = stream;
      next_.store(0);
      err_.store((int)hipSuccess);
      busy_ = WORKERS;
      gen_++;
    }
    wake_.notify_all();
    std::unique_lock<std::mutex> lk(mu_);
    done_.wait(lk, [&] { return busy_ == 0; });
    lk.unlock();
    Relaxed relaxed;
    const hipError_t s = hipStreamSynchronize(stream);  // the pinned chunks are free after it
    *err = err_.load() != (int)hipSuccess ? (hipError_t)err_.load() : s;
    return true;
  }

 private:
  struct Slot {
    void *p = nullptr;
    hipEvent_t ev = nullptr;
  };

  explicit HostCopy(int dev) : dev_(dev) {}

  // Calls of this class stay allowed while another thread captures a graph.
  struct Relaxed {
    hipStreamCaptureMode m = hipStreamCaptureModeRelaxed;
    Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&m); }
    ~Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&m); }
  };

  // The calls of a scope on a device; the caller's current device afterwards.
  struct OnDevice {
    int prev = -1;
    explicit OnDevice(int dev)
    {
      if (hipGetDevice(&prev) != hipSuccess || prev == dev || hipSetDevice(dev) != hipSuccess) prev = -1;
    }
    ~OnDevice()
    {
      if (prev >= 0) (void)hipSetDevice(prev);
    }
  };

  bool start()
  {
    Relaxed relaxed;
    OnDevice here(dev_);  // an event can be recorded on its own device's streams only
    for (Slot &s : slot_)
      if (hipHostMalloc(&s.p, CHUNK, hipHostMallocDefault) != hipSuccess ||
          hipEventCreateWithFlags(&s.ev, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
    for (int w = 0; w < WORKERS; w++) th_[w] = std::thread([this, w] { work(w); });
    return true;
  }

  void fail(hipError_t e)
  {
    if (e != hipSuccess) err_.store((int)e);
  }

  void work(int w)
  {
    (void)hipSetDevice(dev_);
    Relaxed relaxed;
    Slot *s = slot_ + 2 * w;
    unsigned long long seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> lk(mu_);
        wake_.wait(lk, [&] { return stop_ || gen_ != seen; });
        if (stop_) return;
        seen = gen_;
      }
      if (to_device_) upload(s);
      else download(s);
      {
        std::lock_guard<std::mutex> lk(mu_);
        if (--busy_ == 0) done_.notify_one();
      }
    }
  }

  // the next chunk's offset and length; false when none is left or a copy has failed
  bool take(size_t &off, size_t &len)
  {
    off = next_.fetch_add(1) * CHUNK;
    if (off >= bytes_ || err_.load() != (int)hipSuccess) return false;
    len = bytes_ - off < CHUNK ? bytes_ - off : CHUNK;
    return true;
  }

  void upload(Slot *s)
  {
    size_t off, len;
    for (int k = 0; take(off, len); k++) {
      Slot &q = s[k & 1];
      if (k >= 2) fail(hipEventSynchronize(q.ev));
      std::memcpy(q.p, src_ + off, len);
      fail(hipMemcpyAsync(dst_ + off, q.p, len, hipMemcpyHostToDevice, stream_));
      fail(hipEventRecord(q.ev, stream_));
    }
  }

  void download(Slot *s)
  {
    size_t off[2], len[2];
    auto issue = [&](int k) {
      if (!take(off[k], len[k])) return false;
      fail(hipMemcpyAsync(s[k].p, src_ + off[k], len[k], hipMemcpyDeviceToHost, stream_));
      fail(hipEventRecord(s[k].ev, stream_));
      return true;
    };
    bool have = issue(0);
    for (int k = 0; have; k ^= 1) {
      const bool more = issue(k ^ 1);
      fail(hipEventSynchronize(s[k].ev));
      std::memcpy(dst_ + off[k], s[k].p, len[k]);
      have = more;
    }
  }

  const int dev_;
  Slot slot_[2 * WORKERS];
  std::thread th_[WORKERS];
  std::mutex job_, mu_;
  std::condition_variable wake_, done_;
  bool stop_ = false;
  unsigned long long gen_ = 0;
  int busy_ = 0;
  // the current transfer
  char *dst_ = nullptr;
  const char *src_ = nullptr;
  size_t bytes_ = 0;
  bool to_device_ = false;
  hipStream_t stream_ = nullptr;
  std::atomic<size_t> next_{0};
  std::atomic<int> err_{0};
};

// True for memory that the HIP runtime does not know: the caller's ordinary host arrays.  Pinned,
// managed and device memory keeps the plain copy.
inline bool pageable_host(const void *p)
{
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

// The transfers of one context: through the workers of the context's own device, whichever device
// the calling thread has current, or by the plain copy.
class HostTransfers {
 public:
  int device = -1;  // of the context's stream and memory

  // A copy between the caller's host array and device memory, complete on return (ordered behind
  // the work queued on the stream).
  hipError_t copy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t stream) noexcept
  {
    const bool up = kind == hipMemcpyHostToDevice;
    if (bytes >= (up ? HostCopy::MIN_UP : HostCopy::MIN_DOWN) && pageable_host(up ? src : dst)) {
      if (!workers_) {
        moved_ += bytes;
        const bool make = moved_ >= HostCopy::BUILD_BYTES && !refused_;
        workers_ = HostCopy::get(device, make);
        refused_ = refused_ || (make && !workers_);  // no memory or threads for them: not asked for again
      }
      hipError_t e = hipSuccess;
      if (workers_ && workers_->copy(dst, src, bytes, up, stream, &e)) return e;
    }
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, stream);
    return e != hipSuccess ? e : hipStreamSynchronize(stream);
  }

 private:
  std::shared_ptr<HostCopy> workers_;
  bool refused_ = false;
  size_t moved_ = 0;  // bytes of the transfers so far that the workers could have taken
};

}  // namespace fx
