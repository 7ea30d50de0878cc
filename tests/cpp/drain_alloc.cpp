// A download while memory runs out: every allocation in turn fails, in the
// slots, the threads, the events and the lists of pieces (xf_drain.h).  A
// failure has to come out as an exception (the C entry points turn it into a
// status) or as a download with fewer threads, never as an abort, and leaves
// nothing behind.  The HIP calls are stubs in host memory.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

#include "../../xfdtd_cuda_amd/csrc/xf_drain.h"

static std::atomic<long> fail_at{-1}, live{0};
static std::atomic<long> pinned{0}, events{0};

void* operator new(size_t n) {
  if (fail_at.load() >= 0 && fail_at.fetch_sub(1) == 0) throw std::bad_alloc();
  void* p = std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  ++live;
  return p;
}
void operator delete(void* p) noexcept {
  if (p) --live;
  std::free(p);
}
void operator delete(void* p, size_t) noexcept { operator delete(p); }

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n);
  ++pinned;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  --pinned;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(1);
  ++events;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) {
  --events;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
}

// 1: through, 0: bad_alloc
static int download(const std::shared_ptr<xf::StagePool>& pool, const std::vector<double>& from, std::vector<double>& to,
                    size_t all, long k) {
  std::fill(to.begin(), to.end(), 0.0);
  fail_at = k;
  int ok = 1;
  try {
    xf::Drain out(pool, nullptr, 1 << 16, all, size_t(8) << 20);
    if (out.open() != hipSuccess) std::abort();
    const size_t part = from.size() / 8;
    for (size_t q = 0; q < 8; ++q) {
      double* const d = to.data() + q * part;
      if (out.add(from.data() + q * part, part * 8, static_cast<int64_t>(part), 8,
                  [=](const unsigned char* s, int64_t lo, int64_t hi) {
                    std::memcpy(d + lo, s + lo * 8, static_cast<size_t>(hi - lo) * 8);
                  }) != hipSuccess)
        std::abort();
    }
    if (out.finish() != hipSuccess) std::abort();
  } catch (const std::bad_alloc&) {
    ok = 0;
  }
  const bool failed = fail_at.load() < 0 && k >= 0;
  fail_at = -1;
  if (ok && to != from) {
    std::printf("allocation %ld: wrong values\n", k);
    std::exit(1);
  }
  return ok ? (failed ? 2 : 1) : 0;
}

int main() {
  std::vector<double> from(8 * 4096), to(from.size());
  for (size_t q = 0; q < from.size(); ++q) from[q] = static_cast<double>(q) + 0.5;
  for (const size_t all : {size_t(2) << 20, size_t(64) << 20}) {  // ordinary and pinned slots, threads in both
    auto pool = std::make_shared<xf::StagePool>();
    if (download(pool, from, to, all, -1) != 1) return 2;
    const long live0 = live, pinned0 = pinned;
    long k = 0, thrown = 0, fewer = 0;
    for (;; ++k) {
      const int r = download(pool, from, to, all, k);
      if (live != live0 || pinned != pinned0 || events != 0) {
        std::printf("allocation %ld: %ld objects, %ld pinned, %ld events left\n", k, live - live0, pinned - pinned0,
                    events.load());
        return 3;
      }
      if (r == 1) break;  // fewer than k allocations: none failed
      (r == 0 ? thrown : fewer)++;
    }
    std::printf("%zu bytes: %ld allocations, %ld thrown, %ld with fewer threads\n", all, k, thrown, fewer);
    if (thrown == 0 || fewer == 0) return 4;
  }
  return pinned == 0 ? 0 : 5;
}
