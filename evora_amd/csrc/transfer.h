// transfer.h -- host <-> device copies of q in the reference layout, and of
// the potential.
//
// Data crosses PCIe in chunks (chunk_plan) through up to kBuffers pinned host
// buffers, with as much device staging for q.  Per chunk the device runs a
// layout kernel (AoS <-> SoA, given by the caller; the potential needs none)
// and one DMA; a team of host threads, alive for the one transfer, copies
// between the caller's (pageable) array and the pinned buffer.  The host copy
// of one chunk overlaps the DMA and the kernel of the next, so a transfer runs
// at the slower of PCIe (57 GB/s) and host copy instead of their sum plus a
// synchronisation per chunk.  A fresh destination array costs its page faults
// too, which the team shares.  With chunks of up to 64 MB through two buffers
// and 8 threads started for each, and now: up 64^3 (12.6 MB) 0.43 and 0.37 ms,
// 128^3 (101 MB) 2.38 and 2.27, 256^3 (805 MB) 15.35 and 15.48; down into a
// fresh array 48^3 (5.3 MB) 0.32 and 0.26, 64^3 0.69 and 0.53, 128^3 3.24 and
// 2.55, 256^3 17.0 and 16.9.  A 256^3 potential (134 MB) 13.0 ms by one pageable
// copy, 3.5 ms through the buffers.  The pinned buffers are allocated on first
// use (hipHostMalloc).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace evh {

constexpr long long kChunkBytes = 32LL << 20;  // per pinned buffer, at most
constexpr long long kPoolBytes = 64LL << 20;   // all of them
constexpr long long kOnePiece = 10LL << 20;    // an upload of this is one chunk
constexpr int kBuffers = 4;
constexpr long long kCellBytes = 6 * 8;  // one cell of q in the reference layout (6 doubles)

// Threads that copy memory together, for the length of one transfer.
class CopyTeam {
 public:
  // one thread per 8 MB of a transfer of 24 MB or more, 8 at most; if the
  // system gives fewer, those copy it all.  Below that one thread keeps up with
  // most of the link, and where another library's threads spin on every CPU
  // each one more may wait a scheduler's slice of 4 ms: 18 MB after a step loop
  // 2.1 ms against 4.0, 96 MB 13.0 against 16.0 with 12 threads.  Above it more
  // threads show on an idle host too: 30.5 MB down 0.79 ms with three, 1.20
  // with one.
  explicit CopyTeam(size_t total) {
    const unsigned most = std::max(1u, std::min(8u, std::thread::hardware_concurrency()));
    const unsigned n = total < (24u << 20) ? 1u : (unsigned)std::min<size_t>(most, total >> 23);
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

// How a transfer of n units of `bytes` each goes through a pool of `pool`
// bytes: units per chunk and the number of buffers that take turns.  A chunk
// costs a call and a gap on the link (15 us); the first copy of an upload and
// the last of a download have nothing beside them.
// Upload: in one piece up to 10 MB (5.3 MB: 200 us, 215 in two, 255 in five),
// then about the root of the size in MB (12.6 MB: 4 MB; 42 MB: 8 to 12; 805 MB:
// 24 to 32).  Two buffers would do, but it takes the whole pool in equal parts:
// the first touch of its pages, 0.34 ms per MB, then falls to the first upload
// and not to the first download too.
// Download: an eighth, between 1 and 16 MB (5.3 MB: 266 us, 321 in one piece),
// through four buffers where the pool has them: a fresh array takes its page
// faults between the chunks, and they keep the link busy meanwhile (128^3 2.70
// ms with two, 2.5).  Beyond 400 MB the gaps count more: up to 32 MB through two
// (805 MB into a warm array 15.9 ms by 16 MB, 15.5 by 32).
struct ChunkPlan {
  long long units;
  int buffers;
};
inline long long chunk_units(long long n, long long bytes, bool up) {
  const double mb = double(1 << 20), total = double(n) * double(bytes) / mb;
  double chunk;
  if (up) chunk = n * bytes <= kOnePiece ? total : std::min(total / 4, 1.15 * std::sqrt(total));
  else chunk = std::max(1.0, std::min(total / 8, std::max(16.0, total / 24)));
  const long long units = (long long)(std::min(chunk, kChunkBytes / mb) * mb / double(bytes));
  return std::min(std::max(1LL, n), std::max(1LL, units));
}
inline long long pool_bytes(long long max_cells) {
  const auto buffers = [=](bool up, long long turns) {
    const long long units = chunk_units(max_cells, kCellBytes, up);
    return units * std::min(turns, (max_cells + units - 1) / units);
  };
  return std::min(kPoolBytes, kCellBytes * std::max(1LL, std::max(buffers(true, 2), buffers(false, kBuffers))));
}
inline ChunkPlan chunk_plan(long long n, long long bytes, bool up, long long pool) {
  const long long most = pool / bytes;
  long long units = chunk_units(n, bytes, up);
  if (units < n ? 2 * units > most : units > most) units = std::max(1LL, most / 2);
  const long long parts = (2 * most + units) / (2 * units);
  if (up && units < n && parts <= kBuffers) units = most / parts;
  return {units, (int)std::min((long long)kBuffers, most / units)};
}

struct Xfer {
  double *dstage = nullptr;  // device: pool bytes
  char *pinned = nullptr;    // pinned host: as much
  hipEvent_t ev[kBuffers] = {};
  long long pool = 0;

  // device staging for grids of up to max_cells cells
  hipError_t init(long long max_cells) {
    pool = pool_bytes(max_cells);
    hipError_t e = hipMalloc(&dstage, device_bytes());
    for (auto &x : ev)
      if (e == hipSuccess) e = hipEventCreateWithFlags(&x, hipEventDisableTiming);
    return e;
  }
  long long device_bytes() const { return pool; }
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
  // one allocation, on first use; the first touch of its pages takes 0.34 ms
  // per MB, unless the runtime has kept them from an earlier context (64^3
  // context: first upload 2.8 ms with 6 MB that were not kept, 5 ms with 25)
  hipError_t ensure_pinned() {
    return pinned ? hipSuccess : hipHostMalloc((void **)&pinned, pool, hipHostMallocDefault);
  }

  // host q (n cells) -> device; launch(staging, cells, base) enqueues the
  // layout kernel of one chunk on stream s
  template <typename F>
  hipError_t upload(const double *q, long long n, hipStream_t s, F launch) {
    // the first one, which touches the pool, goes through the part of it that
    // downloads use (8.4 MB: 1.9 ms, 3.3 in one piece)
    const bool first = !pinned && n * kCellBytes <= kOnePiece;
    const ChunkPlan c = chunk_plan(n, kCellBytes, !first, pool);
    const long long chunk = c.units;
    hipError_t e = ensure_pinned();
    if (e != hipSuccess) return e;
    CopyTeam team((size_t)(n * kCellBytes));
    long long i = 0;
    for (long long base = 0; base < n; base += chunk, i++) {
      const int b = (int)(i % c.buffers);
      char *const pin = pinned + b * chunk * kCellBytes;
      double *const stage = dstage + 6 * b * chunk;
      const long long cells = std::min(chunk, n - base);
      if (i >= c.buffers && (e = hipEventSynchronize(ev[b])) != hipSuccess) return e;  // pin consumed
      team.copy(pin, q + 6 * base, cells * kCellBytes);
      if ((e = hipMemcpyAsync(stage, pin, cells * kCellBytes, hipMemcpyHostToDevice, s)) != hipSuccess) return e;
      if ((e = hipEventRecord(ev[b], s)) != hipSuccess) return e;
      if ((e = launch(stage, cells, base)) != hipSuccess) return e;
    }
    return hipStreamSynchronize(s);
  }

  // device -> host q (n cells); launch as for upload
  template <typename F>
  hipError_t download(double *q, long long n, hipStream_t s, F launch) {
    const ChunkPlan c = chunk_plan(n, kCellBytes, false, pool);
    return stream_down((char *)q, n, kCellBytes, c, s, [&](int b, long long cells, long long base, const void **src) {
      double *const stage = dstage + 6 * b * c.units;
      *src = stage;
      return launch(stage, cells, base);
    });
  }
  // n doubles at device address d -> host; nothing that writes them is queued
  hipError_t download_doubles(double *out, const double *d, long long n, hipStream_t s) {
    if (n * 8 <= 1 << 20) return hipMemcpy(out, d, n * 8, hipMemcpyDeviceToHost);  // 131 KB 29 us, 41 below; 553 KB 47, 61
    const ChunkPlan c = chunk_plan(n, 8, false, pool);
    return stream_down((char *)out, n, 8, c, s, [&](int, long long, long long base, const void **src) {
      *src = d + base;
      return hipSuccess;
    });
  }

 private:
  // n units of `bytes` -> out; fill(b, units, base, &src) makes a chunk ready
  // on stream s at device address src
  template <typename F>
  hipError_t stream_down(char *out, long long n, long long bytes, const ChunkPlan &c, hipStream_t s, F fill) {
    const long long chunk = c.units, chunks = (n + chunk - 1) / chunk;
    hipError_t e = ensure_pinned();
    if (e != hipSuccess) return e;
    CopyTeam team((size_t)(n * bytes));
    // chunk i is enqueued c.buffers - 1 chunks before it is copied out, into a
    // buffer whose last chunk has been
    for (long long i = 0; i < chunks + c.buffers - 1; i++) {
      if (i < chunks) {
        const int b = (int)(i % c.buffers);
        const long long base = i * chunk, units = std::min(chunk, n - base);
        const void *src = nullptr;
        if ((e = fill(b, units, base, &src)) != hipSuccess) return e;
        if ((e = hipMemcpyAsync(pinned + b * chunk * bytes, src, units * bytes, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
        if ((e = hipEventRecord(ev[b], s)) != hipSuccess) return e;
      }
      const long long j = i - (c.buffers - 1);
      if (j >= 0) {
        const int b = (int)(j % c.buffers);
        const long long base = j * chunk;
        if ((e = hipEventSynchronize(ev[b])) != hipSuccess) return e;
        team.copy(out + base * bytes, pinned + b * chunk * bytes, std::min(chunk, n - base) * bytes);
      }
    }
    return hipSuccess;
  }
};

}  // namespace evh
