// Device to host copies of whole fields into pageable memory.
//
// The runtime stages such a copy through one thread at 10 GB/s: 6.7 ms for the
// 67 MB field of 256 x 128 x 128 cells, as long as 90 of its steps.  The link
// carries five times that, but the host side is a copy, and the first touch of
// a fresh buffer's pages, on one core.  Here several threads, one per processor
// and eight at most, each take chunks of the field, through a pinned slot of
// their own: while one copies out, the others' transfers run.  Memory that is
// pinned already takes the runtime's direct copy.
#include "readback.h"

#include <sched.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>
#include <vector>

namespace lbm {
namespace {

// 268 MB into fresh pages: 25.7 ms by the runtime; 8.9, 7.5 and 7.6 ms with 4, 8
// and 12 threads of 2 MB; 9.2 and 6.8 ms with 8 of 1 and of 4 MB, whose first
// copy costs the more the larger they are.
constexpr int kThreads = 8;
constexpr size_t kSlot = (size_t)2 << 20;
// First copy (slots pinned, threads new) and later ones, ms, by the runtime and
// here: 17 MB 1.7 and 0.95, 2.5 and 0.57; 34 MB 3.8 and 1.9, 2.6 and 1.0; 67 MB
// 6.8 and 6.4, 3.7 and 2.3.  Below the line the first copy would be slower.
constexpr size_t kThreshold = (size_t)32 << 20;

// Whether `p` is memory the runtime does not know, which it stages by itself;
// into memory it has pinned or allocated it copies at the link's rate (67 MB in
// 1.2 ms, 1.8 through the slots, 7.6 the first time).
bool pageable(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

// The processors this process may run on.
int processors() {
  cpu_set_t set;
  return sched_getaffinity(0, sizeof set, &set) == 0 ? std::max(1, CPU_COUNT(&set)) : kThreads;
}

std::mutex g_mu;         // users and staging
std::mutex g_busy;       // one copy at a time has the staging
int g_users = 0;
char* g_slot[kThreads] = {};  // pinned, allocated as copies need them

hipError_t plain(void* dst, const void* src, size_t bytes, hipStream_t s) {
  hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
  return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

}  // namespace

void read_back_retain() {
  std::lock_guard<std::mutex> lk(g_mu);
  g_users++;
}

void read_back_release() {
  std::lock_guard<std::mutex> lk(g_mu);
  if (--g_users > 0) return;
  for (char*& p : g_slot) {
    if (p) (void)hipHostFree(p);
    p = nullptr;
  }
}

hipError_t read_back(void* dst, const void* src, size_t bytes, hipStream_t s) {
  if (bytes < kThreshold || !pageable(dst)) return plain(dst, src, bytes, s);
  std::unique_lock<std::mutex> busy(g_busy, std::try_to_lock);
  if (!busy.owns_lock()) return plain(dst, src, bytes, s);
  const size_t chunks = (bytes + kSlot - 1) / kSlot;
  int threads = (int)std::min<size_t>({(size_t)kThreads, (size_t)processors(), chunks});
  if (threads < 2) return plain(dst, src, bytes, s);  // nothing would overlap
  {
    std::lock_guard<std::mutex> lk(g_mu);
    for (int w = 0; w < threads; w++)
      if (!g_slot[w] && hipHostMalloc((void**)&g_slot[w], kSlot, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        g_slot[w] = nullptr;
        threads = w;
      }
  }
  if (threads == 0) return plain(dst, src, bytes, s);
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipStreamSynchronize(s);  // the threads wait for transfers alone
  if (e != hipSuccess) return e;

  std::atomic<size_t> next{0};
  std::atomic<int> failed{(int)hipSuccess};
  auto work = [&](int w) {
    char* const slot = g_slot[w];
    hipEvent_t done = nullptr;
    hipError_t r = hipSetDevice(dev);
    if (r == hipSuccess) r = hipEventCreateWithFlags(&done, hipEventDisableTiming);
    while (r == hipSuccess && failed.load() == (int)hipSuccess) {
      const size_t k = next.fetch_add(1);
      if (k >= chunks) break;
      const size_t at = k * kSlot, n = std::min(kSlot, bytes - at);
      r = hipMemcpyAsync(slot, static_cast<const char*>(src) + at, n, hipMemcpyDeviceToHost, s);
      if (r == hipSuccess) r = hipEventRecord(done, s);
      if (r == hipSuccess) r = hipEventSynchronize(done);
      if (r == hipSuccess) memcpy(static_cast<char*>(dst) + at, slot, n);
    }
    if (done) (void)hipEventDestroy(done);
    if (r != hipSuccess) failed.store((int)r);
  };
  std::vector<std::thread> others;
  try {
    others.reserve(threads - 1);
    for (int w = 1; w < threads; w++) others.emplace_back(work, w);
  } catch (...) {
    // fewer threads than asked for: those that run and this one share the chunks
  }
  work(0);
  for (std::thread& t : others) t.join();
  e = (hipError_t)failed.load();
  // a transfer into a slot may still run after a failure
  if (e != hipSuccess) (void)hipStreamSynchronize(s);
  return e;
}

hipError_t read_records(double* out, const double* ring, size_t cap, unsigned long long written, size_t take,
                        hipStream_t s) {
  if (take == 0) return hipSuccess;
  const size_t first = (size_t)((written - take) % cap), n = std::min(take, cap - first);
  hipError_t e = hipMemcpyAsync(out, ring + first * 6, n * 48, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess && n < take) e = hipMemcpyAsync(out + n * 6, ring, (take - n) * 48, hipMemcpyDeviceToHost, s);
  return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

}  // namespace lbm
