// Large results to the caller's memory. A pageable destination goes through
// the runtime's single staging thread at about 10 GB/s (a fresh array's pages
// are touched there too); here several threads each bring chunks over into a
// pinned slot of their own and copy them out, so the transfers run back to
// back while the pages are touched in parallel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "internal.hpp"

namespace msim {
namespace {

constexpr size_t kSlotBytes = size_t(2) << 20;
constexpr size_t kMostSlots = 16;     // 32 MiB pinned in the process, at most
constexpr size_t kMostThreads = 8;
// Below this the threads cost more than they save.
constexpr size_t kThreadedBytes = size_t(4) << 20;

// The process's pinned slots: handed out to one download at a time, kept for
// the next, freed with the last context. Held in place, so that handing them
// out and back cannot fail.
class SlotPool {
 public:
  size_t take(void** out, size_t wanted) {
    std::lock_guard<std::mutex> hold(lock_);
    size_t n = 0;
    while (n < wanted) {
      if (kept_ > 0) {
        out[n++] = free_[--kept_];
        continue;
      }
      if (made_ == kMostSlots) break;
      void* ptr = nullptr;
      if (hipHostMalloc(&ptr, kSlotBytes, hipHostMallocPortable) != hipSuccess) {
        static_cast<void>(hipGetLastError());
        break;
      }
      ++made_;
      out[n++] = ptr;
    }
    return n;
  }
  void give(void* const* slots, size_t count) {
    std::lock_guard<std::mutex> hold(lock_);
    for (size_t k = 0; k < count; ++k) free_[kept_++] = slots[k];
    if (users_ == 0) release();
  }
  void enter() {
    std::lock_guard<std::mutex> hold(lock_);
    ++users_;
  }
  void leave() {
    std::lock_guard<std::mutex> hold(lock_);
    if (--users_ == 0) release();
  }

 private:
  void release() {
    made_ -= kept_;
    while (kept_ > 0) static_cast<void>(hipHostFree(free_[--kept_]));
  }
  std::mutex lock_;
  void* free_[kMostSlots] = {};
  size_t kept_ = 0, made_ = 0, users_ = 0;
};

SlotPool g_slots;

// Whether the runtime knows the memory (pinned, managed): the device then
// writes it itself, 67 MB in 1.2 ms and through the slots in 1.8.
bool registered(const void* ptr) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, ptr) != hipSuccess) {
    static_cast<void>(hipGetLastError());
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

}  // namespace

void download_enter() { g_slots.enter(); }
void download_leave() { g_slots.leave(); }

void download(Context& ctx, void* dst, const void* src, size_t bytes, const char* what) {
  auto plain = [&] {
    check(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx.stream), what);
    check(hipStreamSynchronize(ctx.stream), what);
  };
  if (bytes < kThreadedBytes || registered(dst)) return plain();
  const size_t chunks = (bytes + kSlotBytes - 1) / kSlotBytes;
  const size_t cores = std::max<size_t>(std::thread::hardware_concurrency(), 1);
  std::vector<std::thread> threads;
  threads.reserve(kMostThreads);
  void* slots[kMostThreads];
  const size_t count = g_slots.take(slots, std::min({kMostThreads, cores, chunks}));
  if (count < 2) {
    g_slots.give(slots, count);
    return plain();
  }
  // Every chunk is taken by exactly one thread; whatever fails, all are joined
  // and the slots go back only after the stream has drained. Nothing from here
  // to there throws.
  std::atomic<size_t> next{0};
  std::atomic<int> failed{hipSuccess};
  auto work = [&](void* slot) {
    hipEvent_t ready = nullptr;
    hipError_t e = hipSetDevice(ctx.device);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ready, hipEventDisableTiming);
    while (e == hipSuccess && failed.load() == hipSuccess) {
      const size_t c = next.fetch_add(1);
      if (c >= chunks) break;
      const size_t at = c * kSlotBytes, size = std::min(kSlotBytes, bytes - at);
      e = hipMemcpyAsync(slot, static_cast<const char*>(src) + at, size, hipMemcpyDeviceToHost,
                         ctx.stream);
      if (e == hipSuccess) e = hipEventRecord(ready, ctx.stream);
      if (e == hipSuccess) e = hipEventSynchronize(ready);
      if (e == hipSuccess) std::memcpy(static_cast<char*>(dst) + at, slot, size);
    }
    if (ready != nullptr) static_cast<void>(hipEventDestroy(ready));
    if (e != hipSuccess) {
      int none = hipSuccess;
      failed.compare_exchange_strong(none, e);
    }
  };
  try {
    for (size_t k = 1; k < count; ++k) threads.emplace_back(work, slots[k]);
  } catch (const std::exception&) {
    // Fewer threads then (no more of them, or no memory): the others take every
    // chunk.
  }
  work(slots[0]);
  for (auto& t : threads) t.join();
  const hipError_t drained = hipStreamSynchronize(ctx.stream);
  g_slots.give(slots, count);
  check(static_cast<hipError_t>(failed.load()), what);
  check(drained, what);
}

}  // namespace msim
