// Transfers between the caller's pageable memory and the device.
//
// The caller's memory is not pinned, so every byte crosses one pinned buffer on its way.
// Left to the runtime (hipMemcpyAsync on pageable memory) that costs 155 us for 4 MiB up and
// 265 us down (27 and 16 GB/s) where the PCIe link itself takes 76, and 12 to 30 us for a
// few kilobytes.  Here the pinned side is a ring of slots that the host fills or empties
// while the device moves the slots before and after: a transfer is as long as the slower
// of the two, and both sides reach the link's rate --
//  * the device side is a copy kernel that reads or writes the pinned memory directly:
//    sixteen workgroups reach 55 GB/s either way (the most measured with any number), a small
//    copy is 3 us of the stream's time, and nothing waits for another engine;
//  * the host side is memcpy, 28 GB/s on one core for memory that no cache holds, so a large
//    transfer is copied by the calling thread and a few helpers together.
// Measured: experts of 13.2 MB from host memory into HBM 20 -> 42 GB/s (3 matrices each, a wait per
// expert); 3.3 MB of results down 255 -> 95 us; a two-token frame through host buffers 79 -> 59 us.  With an expert's
// matrices in one transfer, chunks as long as the host's lead allows and events only where the ring comes round: eight such
// experts and a token 2870 -> 2600 us (of 1024 x 512 780 -> 645); 1024 x 4096 x 8192 through host buffers 1340 -> 1230.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include <unistd.h>

#include "common.h"

namespace csk {

// Any alignment and size; 16 bytes per lane and access where both sides are aligned.
constexpr int kLinkThreads = 256, kLinkUnroll = 4, kLinkBlocks = 16;
__global__ __launch_bounds__(kLinkThreads) void link_copy_kernel(const unsigned char* __restrict__ src,
                                                                 unsigned char* __restrict__ dst, size_t bytes) {
  const size_t tid = (size_t)blockIdx.x * (kLinkThreads * kLinkUnroll) + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * (kLinkThreads * kLinkUnroll);
  const size_t tid1 = (size_t)blockIdx.x * kLinkThreads + threadIdx.x, stride1 = (size_t)gridDim.x * kLinkThreads;
  size_t done = 0;
  if (((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) == 0) {
    const u32x4* s = reinterpret_cast<const u32x4*>(src);
    u32x4* d = reinterpret_cast<u32x4*>(dst);
    const size_t n = bytes / 16;
    for (size_t i = tid; i < n; i += stride) {
      u32x4 v[kLinkUnroll];
#pragma unroll
      for (int j = 0; j < kLinkUnroll; ++j)
        if (i + (size_t)j * kLinkThreads < n) v[j] = s[i + (size_t)j * kLinkThreads];
#pragma unroll
      for (int j = 0; j < kLinkUnroll; ++j)
        if (i + (size_t)j * kLinkThreads < n) d[i + (size_t)j * kLinkThreads] = v[j];
    }
    done = n * 16;
  } else if (((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 3) == 0) {
    const uint32_t* s = reinterpret_cast<const uint32_t*>(src);
    uint32_t* d = reinterpret_cast<uint32_t*>(dst);
    const size_t n = bytes / 4;
    for (size_t i = tid1; i < n; i += stride1) d[i] = s[i];
    done = n * 4;
  }
  for (size_t i = done + tid1; i < bytes; i += stride1) dst[i] = src[i];
}

constexpr size_t kLinkPiece = (size_t)64 << 10;  // what one thread copies at a time
constexpr size_t kLinkRing = (size_t)16 << 20;

// The calling thread and its helpers copy the pieces of one transfer between the caller's
// memory and the ring, in ascending order; piece i may be taken once `open` is past it.
// Helpers sleep between transfers and while no piece is open -- a result may be behind a long forward --
// after a short spin each time, so that the calls of a loop and the chunks of a running transfer find
// them awake.  They end with the process.
class CopyCrew {
 public:
  static constexpr int kHelpers = 3;
  static constexpr int kSpins = 20000;  // some hundred microseconds

  ~CopyCrew() {
    {
      std::lock_guard<std::mutex> g(m_);
      stop_.store(true);
    }
    cv_.notify_all();
    for (std::thread& t : threads_) t.join();
  }

  // A transfer of up to kParts arrays, one behind the other, each from the beginning of a piece on.  Piece i lies at
  // ring[(at + i * kLinkPiece) % ring_bytes]; `at` is a multiple of a piece.
  static constexpr int kParts = 3;
  struct Job {
    char* host[kParts];
    size_t bytes[kParts];
    long first[kParts + 1];  // piece that a part begins with
    int parts;
    char* ring;
    size_t at, ring_bytes;
    bool up;
    Job(char* ring_, size_t at_, size_t ring_bytes_, bool up_) : parts(0), ring(ring_), at(at_), ring_bytes(ring_bytes_), up(up_) {
      first[0] = 0;
    }
    Job(char* host_, char* ring_, size_t bytes_, size_t at_, size_t ring_bytes_, bool up_) : Job(ring_, at_, ring_bytes_, up_) { add(host_, bytes_); }
    Job() : Job(nullptr, 0, 1, true) {}
    void add(void* h, size_t n) {
      host[parts] = static_cast<char*>(h), bytes[parts] = n;
      first[parts + 1] = first[parts] + (long)((n + kLinkPiece - 1) / kLinkPiece);
      ++parts;
    }
    long pieces() const { return first[parts]; }
    int part_of(long piece) const {
      int p = 0;
      while (piece >= first[p + 1]) ++p;
      return p;
    }
  };

  // false: no memory for the list of pieces.  Helpers that cannot be started are done
  // without: the calling thread takes every piece that nobody else takes.
  bool begin(const Job& j) {
    try {
      if (done_.size() < (size_t)j.pieces()) done_ = std::vector<std::atomic<bool>>((size_t)j.pieces());
    } catch (const std::exception&) {
      return false;
    }
    job_ = j;
    n_ = j.pieces();
    next_.store(0), open_.store(0);
    for (long i = 0; i < n_; ++i) done_[(size_t)i].store(false, std::memory_order_relaxed);
    if (threads_.empty()) {
      const int n = std::min<int>(kHelpers, (int)std::thread::hardware_concurrency() / 4);
      try {
        for (int i = 0; i < n; ++i) threads_.emplace_back([this] { help(); });
      } catch (const std::exception&) {
      }
    }
    {
      std::lock_guard<std::mutex> g(m_);
      running_.store(true);
      epoch_.fetch_add(1);
    }
    cv_.notify_all();
    return true;
  }
  void open_to(long piece) {
    open_.store(std::min(piece, n_));
    wake();
  }
  bool done(long i) const { return done_[(size_t)i].load(std::memory_order_acquire); }
  // takes one open piece, if there is one
  bool work_one() {
    long i = next_.load(std::memory_order_relaxed);
    do {
      if (i >= open_.load(std::memory_order_acquire)) return false;
    } while (!next_.compare_exchange_weak(i, i + 1, std::memory_order_acq_rel));
    const int p = job_.part_of(i);
    const size_t off = (size_t)(i - job_.first[p]) * kLinkPiece, len = std::min(kLinkPiece, job_.bytes[p] - off);
    char* const r = job_.ring + (job_.at + (size_t)i * kLinkPiece) % job_.ring_bytes;
    if (job_.up)
      std::memcpy(r, job_.host[p] + off, len);
    else
      std::memcpy(job_.host[p] + off, r, len);
    done_[(size_t)i].store(true, std::memory_order_release);
    return true;
  }
  // no helper touches the transfer after this; pieces that were never opened stay uncopied
  void end() {
    {
      std::lock_guard<std::mutex> g(m_);
      running_.store(false);
    }
    wake();
    while (inside_.load(std::memory_order_acquire) != 0) relax();
  }

  static void relax() { __builtin_ia32_pause(); }

 private:
  void help() {
    uint64_t seen = 0;
    for (;;) {
      for (int spin = 0; spin < kSpins && epoch_.load(std::memory_order_acquire) == seen && !stop_.load(); ++spin) relax();
      {
        std::unique_lock<std::mutex> g(m_);
        cv_.wait(g, [&] { return stop_.load() || epoch_.load() != seen; });
        if (stop_.load()) return;
        seen = epoch_.load();
        if (!running_.load()) continue;
        inside_.fetch_add(1);
      }
      int spin = 0;
      while (running_.load(std::memory_order_acquire) && next_.load(std::memory_order_relaxed) < n_) {
        if (work_one()) {
          spin = 0;
        } else if (++spin < kSpins) {
          relax();
        } else {
          std::unique_lock<std::mutex> g(m_);
          asleep_.fetch_add(1);  // before the look at open_, as wake() looks after open_ has changed
          cv_.wait(g, [&] { return !running_.load() || next_.load() < open_.load(); });
          asleep_.fetch_sub(1);
          spin = 0;
        }
      }
      inside_.fetch_sub(1, std::memory_order_release);
    }
  }

  void wake() {
    if (asleep_.load() == 0) return;
    { std::lock_guard<std::mutex> g(m_); }  // whoever counts as asleep holds the lock until it waits
    cv_.notify_all();
  }

  std::vector<std::thread> threads_;
  std::mutex m_;
  std::condition_variable cv_;
  std::atomic<bool> stop_{false}, running_{false};
  std::atomic<uint64_t> epoch_{0};
  std::atomic<int> inside_{0}, asleep_{0};
  Job job_{};
  long n_ = 0;
  std::atomic<long> next_{0}, open_{0};
  std::vector<std::atomic<bool>> done_;
};

// What the calling thread does while only the device can get a transfer on: it polls for a while -- a
// chunk takes 20 us -- and leaves longer waits, for the work in front of the transfer, to the runtime.
class DeviceWait {
 public:
  void progress() { polling_ = false; }
  hipError_t once(hipEvent_t e) {
    const auto now = std::chrono::steady_clock::now();
    if (!polling_) since_ = now, polling_ = true;
    if (now - since_ < std::chrono::microseconds(200)) {
      CopyCrew::relax();
      return hipSuccess;
    }
    polling_ = false;
    return hipEventSynchronize(e);
  }

 private:
  bool polling_ = false;
  std::chrono::steady_clock::time_point since_;
};

// The crew of this process.  A forked child has the object but not its threads: joining them, or
// destroying what they sleep on, would wait for ever at its exit, so the child leaves both alone.
class CrewOwner {
 public:
  CrewOwner() = default;
  CrewOwner(const CrewOwner&) = delete;
  CrewOwner& operator=(const CrewOwner&) = delete;
  ~CrewOwner() {
    if (crew_ && pid_ == getpid()) delete crew_;
  }
  bool ready() {
    if (!crew_) crew_ = new (std::nothrow) CopyCrew, pid_ = getpid();
    return crew_ != nullptr;
  }
  CopyCrew* operator->() { return crew_; }

 private:
  CopyCrew* crew_ = nullptr;
  pid_t pid_ = 0;
};

// The pinned ring.  One transfer at a time (the library's lock).
class HostLink {
 public:
  // dst (device) <- host memory, queued on the stream.  The host memory may be reused on return.
  hipError_t to_device(void* dst, const void* host, size_t bytes, hipStream_t st) {
    if (bytes == 0) return hipSuccess;
    const Part part{dst, host, bytes};
    return to_device(&part, 1, st, [](int) { return true; });
  }

  // The same for up to CopyCrew::kParts arrays, none of them empty.  queued(p) is called when the last of part p has been
  // queued, and queues what is to be done with it; false: no more of the transfer.  As a transfer of its own each array
  // began with an empty ring, 20 us in which the device had nothing to do.
  struct Part {
    void* dst;
    const void* host;
    size_t bytes;
  };
  template <class Queued>
  hipError_t to_device(const Part* parts, int n_parts, hipStream_t st, Queued queued) {
    CopyCrew::Job job(ring_, at_, kLinkRing, true);
    for (int p = 0; p < n_parts; ++p) job.add(const_cast<void*>(parts[p].host), parts[p].bytes);
    if (!ready() || (job.ring = ring_, !crew_->begin(job))) {
      for (int p = 0; p < n_parts; ++p) {
        const hipError_t rc = by_runtime(parts[p].dst, parts[p].host, parts[p].bytes, hipMemcpyHostToDevice, st);
        if (rc != hipSuccess || !queued(p)) return rc;
      }
      return hipSuccess;
    }
    hipError_t err = hipSuccess;
    const long n = job.pieces();
    const long first = (long)(at_ / kLinkPiece);
    // Only a transfer that comes round to where it or one before it began has its quarters marked by events: each costs
    // the device 5 us between two copies.  The others leave that to whoever needs their quarters next.
    const bool round = first + n > kPieces;
    long ready_to = 0, sent = 0, opened = 0, want = first == 0 ? 3 : 16;
    int part = 0;
    // A copy kernel costs about 3.5 us of its own.  Onto an idle stream the first ones are short, so that the device starts
    // early; they grow to 1 MiB, and beyond where the host gets ahead: pieces are sent only when the device is about to
    // run out of work, together with all that has been copied by then (chunks of 1 MiB cross the link at 49 GB/s, of 4 at 55).
    using Clock = std::chrono::steady_clock;
    constexpr double kLaunchNs = 15000.0;  // from here to a copy kernel's first bytes, a piece copied in between included
    constexpr double kKernelNs = 3500.0;   // of a copy kernel's own ...
    constexpr double kNsPerByte = 1.0 / 55.0;  // ... and the link's rate
    const auto t0 = Clock::now();
    auto now = [&] { return (double)std::chrono::duration_cast<std::chrono::nanoseconds>(Clock::now() - t0).count(); };
    double busy_until = 0.0;
    DeviceWait wait;
    while (sent < n && err == hipSuccess) {
      while (opened < n) {  // pieces whose place in the ring is free, up to the end of their quarter
        const long end = quarter_end(first + opened);
        // what lay there a round before has been sent, and the device has read it
        if (first + sent < end - kPieces || !free_quarter((int)((end - 1) % kPieces / kPerQuarter), st, err)) break;
        opened = std::min(n, end - first);
        crew_->open_to(opened);
      }
      if (err != hipSuccess) break;
      const bool worked = crew_->work_one();
      while (ready_to < n && ready_to < opened && crew_->done(ready_to)) ++ready_to;
      // up to the end of a quarter of the ring: its event says when it may be filled again
      const long q_end = (round ? quarter_end(first + sent) : kPieces) - first, p_end = job.first[part + 1];
      const long to = std::min(ready_to, std::min(q_end, p_end));
      double t = 0.0;
      if (to > sent && (to == p_end || to == q_end || (to - sent >= want && (t = now()) >= busy_until - kLaunchNs))) {
        const size_t a = (size_t)(sent - job.first[part]) * kLinkPiece;
        const size_t len = std::min(parts[part].bytes, (size_t)(to - job.first[part]) * kLinkPiece) - a;
        err = launch(static_cast<char*>(parts[part].dst) + a, ring_ + (at_ + (size_t)sent * kLinkPiece) % kLinkRing, len, st);
        for (long q = (first + sent) / kPerQuarter; q * kPerQuarter < first + to; ++q) in_use_[q % kQuarters] = true, marked_[q % kQuarters] = false;
        if (err == hipSuccess && round && to == q_end) {
          const int q = (int)((first + sent) % kPieces / kPerQuarter);
          err = hipEventRecord(quarter_[q], st);
          marked_[q] = true;
        }
        busy_until = std::max(t != 0.0 ? t : now(), busy_until) + kKernelNs + (double)len * kNsPerByte;
        sent = to;
        want = std::min(2 * want, 16L);
        if (sent == p_end && err == hipSuccess && !queued(part++)) break;
        wait.progress();
      } else if (worked) {
        wait.progress();
      } else if (sent == opened && opened < n) {  // everything that fits the ring has been sent
        err = wait.once(quarter_[(quarter_end(first + opened) - 1) % kPieces / kPerQuarter]);
      } else {
        CopyCrew::relax();
      }
    }
    crew_->end();
    at_ = (at_ + (size_t)n * kLinkPiece) % kLinkRing;
    return err;
  }

  // host memory <- src (device), after the work queued on the stream.  Waits for all of it.
  hipError_t to_host(void* host, const void* src, size_t bytes, hipStream_t st) {
    if (bytes == 0) return hipSuccess;
    if (!ready()) return by_runtime(host, src, bytes, hipMemcpyDeviceToHost, st);
    hipError_t err = hipSuccess;
    // (places in the ring that an earlier transfer up still reads are written after it, in stream order)
    CopyCrew::Job job(static_cast<char*>(host), ring_, bytes, 0, kLinkRing, false);
    const long n = job.pieces();
    long queued = 0, landed = 0, freed = 0;  // pieces requested, in pinned memory, copied out
    long ends[kDown];
    int put = 0, got = 0;  // chunks requested and landed
    if (!crew_->begin(job)) return by_runtime(host, src, bytes, hipMemcpyDeviceToHost, st);
    DeviceWait wait;
    while (freed < n && err == hipSuccess) {
      // Half of what is left per chunk, at most 4 MiB and at least 512 KiB: few chunks (each costs about 9 us for
      // its kernel and event, half of what a MiB takes), and little left to copy once the last has landed.
      while (queued < n && put - got < kDown && err == hipSuccess) {
        long len = std::max(8L, std::min(64L, (n - queued + 1) / 2));
        len = std::min(len, n - queued);
        const long to_wrap = kPieces - queued % kPieces;
        len = std::min(len, to_wrap);
        if (queued + len > freed + kPieces) break;
        const size_t a = (size_t)queued * kLinkPiece, cb = std::min(bytes, (size_t)(queued + len) * kLinkPiece) - a;
        err = launch(ring_ + a % kLinkRing, static_cast<const char*>(src) + a, cb, st);
        if (err == hipSuccess) err = hipEventRecord(down_[put % kDown], st);
        queued += len;
        ends[put++ % kDown] = queued;
      }
      while (got < put && err == hipSuccess) {
        const hipError_t rc = hipEventQuery(down_[got % kDown]);
        if (rc == hipErrorNotReady) {
          (void)hipGetLastError();
          break;
        }
        err = rc;
        landed = ends[got++ % kDown];
        crew_->open_to(landed);
      }
      if (crew_->work_one())
        wait.progress();
      else if (freed == landed && got < put && err == hipSuccess)
        err = wait.once(down_[got % kDown]);
      else
        CopyCrew::relax();
      while (freed < landed && crew_->done(freed)) ++freed;
    }
    crew_->end();
    idle();
    return err;
  }

  // the stream is known to be idle: the whole ring is free
  void idle() {
    at_ = 0;
    for (bool& b : in_use_) b = false;
  }

 private:
  static constexpr long kPieces = (long)(kLinkRing / kLinkPiece);
  static constexpr int kQuarters = 4;
  static constexpr long kPerQuarter = kPieces / kQuarters;
  static constexpr int kDown = 8;  // chunks on their way down at once
  char* ring_ = nullptr;
  size_t at_ = 0;  // where the next transfer up starts
  hipEvent_t quarter_[kQuarters] = {}, down_[kDown] = {};
  bool in_use_[kQuarters] = {};  // the device may still be reading that quarter
  bool marked_[kQuarters] = {};  // and its event comes behind the last copy that does
  CrewOwner crew_;
  bool refused_ = false;

  // false: the machine gives no pinned memory (asked for once), or no memory for the crew
  bool ready() {
    if (ring_) return true;
    if (refused_ || !crew_.ready()) return false;
    hipError_t rc = hipSuccess;
    for (hipEvent_t* e = quarter_; e < quarter_ + kQuarters && rc == hipSuccess; ++e)
      if (!*e) rc = hipEventCreateWithFlags(e, hipEventDisableTiming);
    for (hipEvent_t* e = down_; e < down_ + kDown && rc == hipSuccess; ++e)
      if (!*e) rc = hipEventCreateWithFlags(e, hipEventDisableTiming);
    if (rc == hipSuccess) rc = hipHostMalloc(reinterpret_cast<void**>(&ring_), kLinkRing, hipHostMallocDefault);
    if (rc == hipSuccess) return true;
    (void)hipGetLastError();
    ring_ = nullptr, refused_ = true;
    return false;
  }
  // The runtime's own copy of pageable memory, with the same promise: the host's side is done on return.
  hipError_t by_runtime(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t st) {
    const hipError_t rc = hipMemcpyAsync(dst, src, bytes, kind, st);
    const hipError_t rs = hipStreamSynchronize(st);
    if (rc == hipSuccess && rs == hipSuccess) idle();
    return rc != hipSuccess ? rc : rs;
  }
  static long quarter_end(long piece) { return (piece / kPerQuarter + 1) * kPerQuarter; }
  static hipError_t launch(void* dst, const void* src, size_t bytes, hipStream_t st) {
    const size_t per_block = (size_t)kLinkThreads * kLinkUnroll * 16;
    const unsigned blocks = (unsigned)std::min<size_t>(kLinkBlocks, std::max<size_t>(1, (bytes + per_block - 1) / per_block));
    link_copy_kernel<<<dim3(blocks), kLinkThreads, 0, st>>>(static_cast<const unsigned char*>(src), static_cast<unsigned char*>(dst), bytes);
    return hipGetLastError();
  }
  bool free_quarter(int q, hipStream_t st, hipError_t& err) {
    if (!in_use_[q]) return true;
    if (!marked_[q]) {
      err = hipEventRecord(quarter_[q], st);
      if (err != hipSuccess) return false;
      marked_[q] = true;
    }
    const hipError_t rc = hipEventQuery(quarter_[q]);
    if (rc == hipErrorNotReady) {
      (void)hipGetLastError();
      return false;
    }
    in_use_[q] = false;
    err = rc;
    return rc == hipSuccess;
  }
};

}  // namespace csk
