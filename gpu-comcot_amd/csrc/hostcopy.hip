// Reading planes back.  hipMemcpy into ordinary memory stages through a
// pinned buffer of its own and copies out with one thread; where the pages
// are fresh, as a newly allocated output array's, that thread also takes
// every page fault: 50 MB in 4.7 ms (huge pages) to 12 ms, 3.1 ms with the
// pages there, against 0.9 ms that the link needs.  Here the transfers run
// ahead through a ring of pinned slots and several threads copy out, faults
// included.
#include "hostcopy.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace gc {

namespace {

// Measured into fresh huge pages, 12.6 and 50.3 MB (hipMemcpy 0.97, 4.7 ms):
// slots of 2 MB, 6 of them, 4 threads 0.60, 1.69; 8 and 6 threads 0.59, 1.55;
// 1 MB, 6 and 4 0.60, 1.91; 4 MB, 4 and 4 0.72, 1.93; 512 KB, 12 and 6 0.69,
// 2.43.  3 - 4 MB take the same time either way, and taking the ring and
// giving it back cost 0.8 ms, so planes from 8 MB use it.
constexpr size_t kSlot = 2u << 20;
constexpr int kSlots = 6, kThreads = 4;
constexpr size_t kStagedMin = 8u << 20;

std::mutex g_mutex;  // one copy at a time uses the ring
char *g_ring = nullptr;
hipEvent_t g_done[kSlots];

hipError_t ring() {
  if (g_ring) return hipSuccess;
  int n = 0;
  hipError_t e = hipSuccess;
  while (n < kSlots && (e = hipEventCreateWithFlags(&g_done[n], hipEventDisableTiming)) == hipSuccess) ++n;
  void *p = nullptr;
  if (e == hipSuccess) e = hipHostMalloc(&p, kSlots * kSlot, hipHostMallocDefault);
  if (e != hipSuccess)
    while (n > 0) (void)hipEventDestroy(g_done[--n]);
  g_ring = static_cast<char *>(p);
  return e;
}

// Memory that HIP does not know: threads may write it.  Pinned, managed and
// device memory (and null) are hipMemcpy's.
bool ordinary(const void *p) {
  hipPointerAttribute_t a;
  if (!p) return false;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

}  // namespace

void copy_release() {
  std::lock_guard<std::mutex> lock(g_mutex);
  if (!g_ring) return;
  for (hipEvent_t e : g_done) (void)hipEventDestroy(e);
  (void)hipHostFree(g_ring);
  g_ring = nullptr;
}

hipError_t copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t st) {
  const unsigned cpus = std::thread::hardware_concurrency();
  std::unique_lock<std::mutex> lock(g_mutex, std::defer_lock);
  if (bytes >= kStagedMin && cpus >= 4 && ordinary(dst)) lock.lock();
  if (!lock.owns_lock() || ring() != hipSuccess) {
    if (lock.owns_lock()) (void)hipGetLastError();
    const hipError_t e = hipStreamSynchronize(st);
    return e != hipSuccess ? e : hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
  }
  const size_t n = (bytes + kSlot - 1) / kSlot;
  auto part = [&](size_t c) { return std::min(kSlot, bytes - c * kSlot); };
  std::atomic<size_t> arrived{0}, next{0};  // chunks in the ring so far; next to copy out
  std::atomic<bool> stop{false};
  std::atomic<size_t> emptied[kSlots] = {};  // chunks up to this one have left the slot
  auto work = [&] {
    for (size_t c; (c = next.fetch_add(1)) < n;) {
      while (arrived.load(std::memory_order_acquire) <= c) {
        if (stop.load()) return;
        std::this_thread::yield();
      }
      std::memcpy(static_cast<char *>(dst) + c * kSlot, g_ring + c % kSlots * kSlot, part(c));
      emptied[c % kSlots].store(c + 1, std::memory_order_release);
    }
  };
  std::thread team[kThreads];
  int hands = 0;
  try {
    for (; hands < kThreads; ++hands) team[hands] = std::thread(work);
  } catch (const std::exception &) {  // no more threads: those that started do it
  }
  hipError_t e = hipSuccess;
  size_t sent = 0;
  for (size_t c = 0; c < n && e == hipSuccess && hands > 0; ++c) {
    // keep the ring full; a chunk waits for the one that held its slot
    while (e == hipSuccess && sent < n && sent < c + kSlots) {
      const size_t before = sent < kSlots ? 0 : sent - kSlots + 1;
      if (emptied[sent % kSlots].load(std::memory_order_acquire) < before) {
        if (sent > c) break;  // meanwhile chunk c may arrive
        std::this_thread::yield();
        continue;
      }
      e = hipMemcpyAsync(g_ring + sent % kSlots * kSlot, static_cast<const char *>(src) + sent * kSlot,
                         part(sent), hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipEventRecord(g_done[sent % kSlots], st);
      ++sent;
    }
    if (e == hipSuccess) e = hipEventSynchronize(g_done[c % kSlots]);
    if (e == hipSuccess) arrived.store(c + 1, std::memory_order_release);
  }
  if (e != hipSuccess) stop.store(true);
  for (int k = 0; k < hands; ++k) team[k].join();
  if (e != hipSuccess) (void)hipStreamSynchronize(st);  // nothing may still write the ring
  if (hands == 0) {
    e = hipStreamSynchronize(st);
    if (e == hipSuccess) e = hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
  }
  return e;
}

}  // namespace gc
