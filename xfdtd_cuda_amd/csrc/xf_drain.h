// xf_drain.h -- device arrays on their way into the caller's host arrays.
//
// A download reads the state through two staging slots by turns: while the
// copy engine fills one, the host's threads convert the other into the
// caller's arrays.  A copy into the caller's own (pageable) memory, and the
// one large buffer a component was unpacked from before, ran at 9 GB/s, the
// buffer's zeroing and page faults included: 536^3 FP64 790 ms, now 182 ms
// (41 GB/s); a batch's 8 grids in FP32 76 ms, now 25.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <exception>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace xf {

// Pinned slots that the engines of a process share: at most kKept pairs are
// kept between downloads, and the last engine to go gives them back.
class StagePool {
 public:
  static constexpr size_t kSlot = size_t(16) << 20;
  StagePool() { free_.reserve(kKept); }  // give() allocates nothing
  static std::shared_ptr<StagePool> shared() {
    static std::mutex m;
    static std::weak_ptr<StagePool> pool;
    std::lock_guard<std::mutex> lock(m);
    std::shared_ptr<StagePool> p = pool.lock();
    if (!p) pool = p = std::make_shared<StagePool>();
    return p;
  }
  ~StagePool() {
    for (void* p : free_) (void)hipHostFree(p);
  }
  // two slots of kSlot bytes, or null (the caller then takes ordinary memory)
  void* take() {
    {
      std::lock_guard<std::mutex> lock(m_);
      if (!free_.empty()) {
        void* p = free_.back();
        free_.pop_back();
        return p;
      }
    }
    void* p = nullptr;
    if (hipHostMalloc(&p, 2 * kSlot, hipHostMallocPortable) == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
  }
  void give(void* p) {
    {
      std::lock_guard<std::mutex> lock(m_);
      if (free_.size() < kKept) {
        free_.push_back(p);
        return;
      }
    }
    (void)hipHostFree(p);
  }

 private:
  static constexpr size_t kKept = 2;
  std::mutex m_;
  std::vector<void*> free_;
};

// Threads that work through numbered units together with the caller.
class Crew {
 public:
  explicit Crew(int n) {
    try {
      threads_.reserve(static_cast<size_t>(n));
      for (int q = 1; q < n; ++q) threads_.emplace_back([this] { loop(); });
    } catch (const std::exception&) {
      // no thread or no memory for one: fewer threads
    }
  }
  ~Crew() {
    {
      std::lock_guard<std::mutex> lock(m_);
      stop_ = true;
    }
    go_.notify_all();
    for (std::thread& t : threads_) t.join();
  }
  void run(size_t units, const std::function<void(size_t)>& fn) {
    {
      std::lock_guard<std::mutex> lock(m_);
      fn_ = &fn;
      units_ = units;
      next_ = 0;
      busy_ = threads_.size();
      ++turn_;
    }
    go_.notify_all();
    work();
    std::unique_lock<std::mutex> lock(m_);
    done_.wait(lock, [this] { return busy_ == 0; });
  }

 private:
  void work() {
    for (size_t u; (u = next_.fetch_add(1)) < units_;) (*fn_)(u);
  }
  void loop() {
    uint64_t seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> lock(m_);
        go_.wait(lock, [&] { return stop_ || turn_ != seen; });
        if (stop_) return;
        seen = turn_;
      }
      work();
      std::lock_guard<std::mutex> lock(m_);
      if (--busy_ == 0) done_.notify_one();
    }
  }
  std::vector<std::thread> threads_;
  std::mutex m_;
  std::condition_variable go_, done_;
  const std::function<void(size_t)>* fn_ = nullptr;
  size_t units_ = 0, busy_ = 0;
  std::atomic<size_t> next_{0};
  uint64_t turn_ = 0;
  bool stop_ = false;
};

// One download.  add() queues a copy; put(from, lo, hi) then converts rows
// [lo, hi) of it.  The rows of one add must be convertible in any order.
class Drain {
 public:
  using Put = std::function<void(const unsigned char*, int64_t, int64_t)>;

  // most: the largest piece that cannot be cut; all: bytes in total; work: the
  // conversion, in bytes of the caller's memory that a copy writes as fast.
  Drain(std::shared_ptr<StagePool> pool, hipStream_t stream, size_t most, size_t all, size_t work)
      : pool_(std::move(pool)), stream_(stream) {
    // what may throw comes before the slots, which only the destructor gives back
    const int cpus = std::max(1, static_cast<int>(std::thread::hardware_concurrency()));
    // a thread's start is worth it from about 2 MiB of conversion on
    crew_ = std::make_unique<Crew>(static_cast<int>(
        std::min<size_t>(std::min(cpus, 16), std::max<size_t>(1, work / (size_t(2) << 20)))));
    // Pinning two slots takes 0.3 to 1.5 ms, the first time in a process, which a
    // download pays back from about kPinFrom bytes on; a smaller one goes through
    // ordinary memory, where 20 to 40 MB took 7 to 10 ms (in pinned slots 1.1 to
    // 2).  A download of up to 64 MiB fills four slots, so that copies and
    // conversion overlap.
    if (all >= kPinFrom && most <= StagePool::kSlot) pinned_ = pool_->take();
    slot_ = pinned_ ? std::max(most, std::min(std::max(all / 4, size_t(1) << 20), StagePool::kSlot))
                    : std::max(most, std::min(all, StagePool::kSlot));
    base_ = static_cast<unsigned char*>(pinned_ ? pinned_ : std::malloc(2 * slot_));
  }
  ~Drain() {
    for (hipEvent_t& e : event_)
      if (e) (void)hipEventDestroy(e);
    if (queued_) (void)hipStreamSynchronize(stream_);  // an error left copies in flight
    if (pinned_)
      pool_->give(pinned_);
    else
      std::free(base_);
  }
  Drain(const Drain&) = delete;
  Drain& operator=(const Drain&) = delete;

  hipError_t open() {
    if (!base_) return hipErrorOutOfMemory;
    for (hipEvent_t& e : event_) {
      const hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
      if (r != hipSuccess) return r;
    }
    return hipSuccess;
  }
  size_t slot_bytes() const { return slot_; }

  // bytes at dev: `rows` rows to convert, row_bytes of the caller's memory each
  hipError_t add(const void* dev, size_t bytes, int64_t rows, size_t row_bytes, Put put) {
    if (bytes == 0 || rows == 0) return hipSuccess;
    if (bytes > slot_) return hipErrorInvalidValue;
    if (used_ + bytes > slot_) {
      const hipError_t r = flush();
      if (r != hipSuccess) return r;
    }
    unsigned char* const at = base_ + cur_ * slot_ + used_;
    const hipError_t r = hipMemcpyAsync(at, dev, bytes, hipMemcpyDeviceToHost, stream_);
    if (r != hipSuccess) return r;
    queued_ = true;
    const int64_t step = std::max<int64_t>(1, static_cast<int64_t>(kUnit / std::max<size_t>(1, row_bytes)));
    const size_t piece = pieces_[cur_].size();
    pieces_[cur_].push_back({at, std::move(put)});
    for (int64_t lo = 0; lo < rows; lo += step) units_[cur_].push_back({piece, lo, std::min(rows, lo + step)});
    used_ += (bytes + 63) / 64 * 64;
    return hipSuccess;
  }
  hipError_t finish() {
    for (int q = 0; q < 2; ++q) {
      const hipError_t r = flush();
      if (r != hipSuccess) return r;
    }
    queued_ = false;
    return hipSuccess;
  }

 private:
  struct Piece {
    const unsigned char* from;
    Put put;
  };
  struct Unit {
    size_t piece;
    int64_t lo, hi;
  };
  // the slot being filled is closed, the other one converted and opened
  hipError_t flush() {
    if (!pieces_[cur_].empty()) {
      const hipError_t r = hipEventRecord(event_[cur_], stream_);
      if (r != hipSuccess) return r;
    }
    cur_ ^= 1;
    used_ = 0;
    if (pieces_[cur_].empty()) return hipSuccess;
    const hipError_t r = hipEventSynchronize(event_[cur_]);
    if (r != hipSuccess) return r;
    const std::vector<Unit>& units = units_[cur_];
    const std::vector<Piece>& pieces = pieces_[cur_];
    crew_->run(units.size(), [&](size_t u) {
      const Piece& p = pieces[units[u].piece];
      p.put(p.from, units[u].lo, units[u].hi);
    });
    pieces_[cur_].clear();
    units_[cur_].clear();
    return hipSuccess;
  }

  static constexpr size_t kPinFrom = size_t(4) << 20, kUnit = size_t(256) << 10;
  std::shared_ptr<StagePool> pool_;
  hipStream_t stream_;
  void* pinned_ = nullptr;
  unsigned char* base_ = nullptr;
  size_t slot_ = 0, used_ = 0;
  int cur_ = 0;
  bool queued_ = false;
  hipEvent_t event_[2]{};
  std::vector<Piece> pieces_[2];
  std::vector<Unit> units_[2];
  std::unique_ptr<Crew> crew_;
};

}  // namespace xf
