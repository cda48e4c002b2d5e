// transfer.h -- host <-> device copies of q in the reference layout, and of
// the potential.
//
// Data crosses PCIe in chunks of at most kChunkBytes through kBuffers pinned
// host buffers, with as many device staging buffers for q.  Per chunk the
// device runs a layout kernel (AoS <-> SoA, given by the caller; the potential
// needs none) and one DMA; a team of host threads, alive for the one transfer,
// copies between the caller's (pageable) array and the pinned buffer.  The
// host copy of one chunk overlaps the DMA and the kernel of the next, so a
// transfer runs at the slower of PCIe and host copy instead of their sum plus
// a synchronisation per chunk.  A fresh destination array costs its page
// faults too, which the team shares.  Into a fresh array: 256^3 (805 MB) 18.2 ms
// with 8 threads started for each chunk of 64 MB, 17.2 ms now (47 GB/s; the
// link gives 57); its potential (134 MB) 13.0 ms by one pageable copy, 3.5 ms
// now; 64^3 (12.6 MB) 0.66 and 0.56 ms.  The pinned buffers are
// allocated on first use (hipHostMalloc).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace evh {

constexpr long long kChunkBytes = 16LL << 20;  // per pinned buffer
constexpr int kBuffers = 4;
constexpr long long kCellBytes = 6 * 8;  // one cell of q in the reference layout (6 doubles)

// Threads that copy memory together, for the length of one transfer.
class CopyTeam {
 public:
  // one thread per 8 MB of a transfer of 32 MB or more, 8 at most; if the
  // system gives fewer, those copy it all.  More threads are no faster on an
  // idle host (64^3, 12.6 MB: 0.57 ms either way; 128^3 2.66 and 2.67 ms with one per
  // 2 MB, 16 at most), and where another library's threads spin on every CPU
  // each one may wait a scheduler's slice of 4 ms: 18 MB after a step loop
  // 2.1 ms against 4.0, 96 MB 13.0 against 16.0.
  explicit CopyTeam(size_t total) {
    const unsigned most = std::max(1u, std::min(8u, std::thread::hardware_concurrency()));
    const unsigned n = total < (32u << 20) ? 1u : (unsigned)std::min<size_t>(most, total >> 23);
    try {
      for (unsigned i = 1; i < n; i++) threads_.emplace_back([this, i] { work(i); });
    } catch (const std::exception &) {
    }
  }
  ~CopyTeam() {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      stop_ = true;
    }
    start_.notify_all();
    for (auto &t : threads_) t.join();
  }
  CopyTeam(const CopyTeam &) = delete;
  CopyTeam &operator=(const CopyTeam &) = delete;

  void copy(void *dst, const void *src, size_t bytes) {
    if (threads_.empty() || bytes < (1u << 20)) {
      std::memcpy(dst, src, bytes);
      return;
    }
    {
      std::lock_guard<std::mutex> lock(mutex_);
      dst_ = (char *)dst;
      src_ = (const char *)src;
      bytes_ = bytes;
      left_ = (unsigned)threads_.size();
      job_++;
    }
    start_.notify_all();
    part(0);
    std::unique_lock<std::mutex> lock(mutex_);
    done_.wait(lock, [this] { return left_ == 0; });
  }

 private:
  void part(unsigned i) {
    const size_t n = threads_.size() + 1, step = (bytes_ / n + 4096) & ~size_t(4095);
    const size_t off = i * step;
    if (off < bytes_) std::memcpy(dst_ + off, src_ + off, std::min(step, bytes_ - off));
  }
  void work(unsigned i) {
    unsigned seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> lock(mutex_);
        start_.wait(lock, [&] { return stop_ || job_ != seen; });
        if (stop_) return;
        seen = job_;
      }
      part(i);
      std::lock_guard<std::mutex> lock(mutex_);
      if (--left_ == 0) done_.notify_one();
    }
  }

  std::vector<std::thread> threads_;
  std::mutex mutex_;
  std::condition_variable start_, done_;
  char *dst_ = nullptr;
  const char *src_ = nullptr;
  size_t bytes_ = 0;
  unsigned job_ = 0, left_ = 0;
  bool stop_ = false;
};

struct Xfer {
  double *dstage = nullptr;            // device: buffers * chunk_cells * 6 doubles
  char *pinned = nullptr;              // pinned host: as much
  hipEvent_t ev[kBuffers] = {};
  long long chunk_cells = 0, buffers = 0;  // chunks of the largest grid fill up to kBuffers of them

  // device staging for grids of up to max_cells cells: the buffers hold the
  // largest chunk that chunk_units gives
  hipError_t init(long long max_cells) {
    chunk_cells = kChunkBytes / kCellBytes;
    chunk_cells = std::min(std::max(1LL, max_cells), chunk_units(max_cells, kCellBytes));
    buffers = std::min((long long)kBuffers, (max_cells + chunk_cells - 1) / chunk_cells);
    hipError_t e = hipMalloc(&dstage, device_bytes());
    for (auto &x : ev)
      if (e == hipSuccess) e = hipEventCreateWithFlags(&x, hipEventDisableTiming);
    return e;
  }
  long long device_bytes() const { return buffers * chunk_cells * kCellBytes; }
  void release() {
    if (dstage) (void)hipFree(dstage);
    if (pinned) (void)hipHostFree(pinned);
    pinned = nullptr;
    for (auto &x : ev) {
      if (x) (void)hipEventDestroy(x);
      x = nullptr;
    }
    dstage = nullptr;
  }
  // one allocation, of what a transfer can turn over: pinning takes 0.1 ms and
  // more each time (64^3 context: first upload 0.9 ms with four buffers of the
  // whole state's size, 0.6 ms with these; 128^2 0.13 -> 0.09)
  hipError_t ensure_pinned() {
    return pinned ? hipSuccess : hipHostMalloc((void **)&pinned, device_bytes(), hipHostMallocDefault);
  }
  char *pin(int b) const { return pinned + (long long)b * kCellBytes * chunk_cells; }
  double *stage(int b) const { return dstage + (long long)b * 6 * chunk_cells; }

  // units of `bytes` each per chunk for a transfer of n: an eighth of it, so
  // that small ones overlap too, between 1 MB and the buffer
  long long chunk_units(long long n, long long bytes) const {
    const long long most = chunk_cells * kCellBytes / bytes;
    return std::max(1LL, std::min(most, std::max((1LL << 20) / bytes, (n + 7) / 8)));
  }

  // host q (n cells) -> device; launch(staging, cells, base) enqueues the
  // layout kernel of one chunk on stream s
  template <typename F>
  hipError_t upload(const double *q, long long n, hipStream_t s, F launch) {
    const long long chunk = chunk_units(n, kCellBytes);
    hipError_t e = ensure_pinned();
    if (e != hipSuccess) return e;
    CopyTeam team((size_t)(n * kCellBytes));
    long long i = 0;
    for (long long base = 0; base < n; base += chunk, i++) {
      const int b = (int)(i % kBuffers);
      const long long cells = std::min(chunk, n - base);
      if (i >= kBuffers && (e = hipEventSynchronize(ev[b])) != hipSuccess) return e;  // pin(b) consumed
      team.copy(pin(b), q + 6 * base, cells * kCellBytes);
      if ((e = hipMemcpyAsync(stage(b), pin(b), cells * kCellBytes, hipMemcpyHostToDevice, s)) != hipSuccess) return e;
      if ((e = hipEventRecord(ev[b], s)) != hipSuccess) return e;
      if ((e = launch(stage(b), cells, base)) != hipSuccess) return e;
    }
    return hipStreamSynchronize(s);
  }

  // device -> host q (n cells); launch as for upload
  template <typename F>
  hipError_t download(double *q, long long n, hipStream_t s, F launch) {
    return stream_down((char *)q, n, kCellBytes, s, [&](int b, long long cells, long long base, const void **src) {
      *src = stage(b);
      return launch(stage(b), cells, base);
    });
  }
  // n doubles at device address d -> host
  hipError_t download_doubles(double *out, const double *d, long long n, hipStream_t s) {
    return stream_down((char *)out, n, 8, s, [&](int, long long, long long base, const void **src) {
      *src = d + base;
      return hipSuccess;
    });
  }

 private:
  // n units of `bytes` -> out; fill(b, units, base, &src) makes a chunk ready
  // on stream s at device address src
  template <typename F>
  hipError_t stream_down(char *out, long long n, long long bytes, hipStream_t s, F fill) {
    const long long chunk = chunk_units(n, bytes), chunks = (n + chunk - 1) / chunk;
    hipError_t e = ensure_pinned();
    if (e != hipSuccess) return e;
    CopyTeam team((size_t)(n * bytes));
    // chunk i is enqueued kBuffers - 1 chunks before it is copied out, into a
    // buffer whose last chunk has been
    for (long long i = 0; i < chunks + kBuffers - 1; i++) {
      if (i < chunks) {
        const int b = (int)(i % kBuffers);
        const long long base = i * chunk, units = std::min(chunk, n - base);
        const void *src = nullptr;
        if ((e = fill(b, units, base, &src)) != hipSuccess) return e;
        if ((e = hipMemcpyAsync(pin(b), src, units * bytes, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
        if ((e = hipEventRecord(ev[b], s)) != hipSuccess) return e;
      }
      const long long j = i - (kBuffers - 1);
      if (j >= 0) {
        const int b = (int)(j % kBuffers);
        const long long base = j * chunk;
        if ((e = hipEventSynchronize(ev[b])) != hipSuccess) return e;
        team.copy(out + base * bytes, pin(b), std::min(chunk, n - base) * bytes);
      }
    }
    return hipSuccess;
  }
};

}  // namespace evh
