// copy_ring.hpp -- large results to host arrays through a ring of pinned slots that
// several threads empty (host code; Api: the device's copies, events and pinned memory).
//
// The runtime's copy to pageable memory is bound by one thread reading the staging
// memory the GPU has just written (about 16 GB/s, where the link gives 50).  Here
// kThreads threads empty the slots while the next chunks are on the way: 48 MB of
// stresses and strains with the assembly that precedes them take 1.83 ms against 3.15 ms
// (1.88 ms with 2 threads, 2.2 to 2.3 ms with 1 MB chunks and 4 to 8 threads, each array
// for itself).
#pragma once

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

namespace onsas {

struct CopyPart {
  void* dst;
  const void* src;  // on the device
  size_t bytes;
};

// Api: Event; bool pinned(char**, size_t), free_pinned(char*), make(Event*),
// destroy(Event); bool queue(char* pinned, const void* src, size_t), record(Event),
// wait(Event), from any thread; drain()
template <typename Api, size_t kChunkBytes = size_t(2) << 20, int kSlots = 8, int kThreads = 4>
class CopyRing {
 public:
  static constexpr size_t kChunk = kChunkBytes;
  static_assert(kSlots % kThreads == 0, "a slot belongs to one thread");
  // kNone: nothing has been queued (no pinned memory, events, host memory or threads to be
  // had); kFailed: a copy failed, the arrays hold anything
  enum Result { kDone, kNone, kFailed };

  Result copy(Api& api, const std::vector<CopyPart>& parts) {
    std::vector<CopyPart> chunks;
    std::vector<std::thread> threads;
    std::atomic<int64_t> issued{0};      // chunks whose transfer is queued
    std::atomic<int64_t> taken[kSlots];  // per slot: chunks copied out of it
    for (auto& q : taken) q = 0;
    std::atomic<bool> failed{false};
    // chunk i lives in slot i % kSlots and belongs to thread i % kThreads
    auto work = [&](int w) {
      for (int64_t i = w; i < (int64_t)chunks.size(); i += kThreads) {
        while (issued.load(std::memory_order_acquire) <= i && !failed) std::this_thread::yield();
        if (failed) return;
        const int k = (int)(i % kSlots);
        if (!api.wait(ev_[k])) {
          failed = true;
          return;
        }
        std::memcpy(chunks[i].dst, mem_ + k * kChunk, chunks[i].bytes);
        taken[k].fetch_add(1, std::memory_order_release);
      }
    };
    bool ready = make(api);
    try {
      for (const CopyPart& p : parts)
        for (size_t o = 0; ready && o < p.bytes; o += kChunk)
          chunks.push_back({(char*)p.dst + o, (const char*)p.src + o, std::min(kChunk, p.bytes - o)});
      threads.reserve(kThreads);
      for (int w = 0; ready && w < kThreads; ++w) threads.emplace_back(work, w);
    } catch (...) {
      ready = false;
    }
    bool ok = true;
    for (int64_t i = 0; ready && ok && i < (int64_t)chunks.size(); ++i) {
      const int k = (int)(i % kSlots);
      while (taken[k].load(std::memory_order_acquire) < i / kSlots && !failed) std::this_thread::yield();
      if (failed) break;  // the slot may still be read
      ok = api.queue(mem_ + k * kChunk, chunks[i].src, chunks[i].bytes) && api.record(ev_[k]);
      if (ok) issued.store(i + 1, std::memory_order_release);
    }
    const bool bad = !ok || failed;
    if (!ready || bad) failed = true;  // the threads leave
    for (auto& t : threads) t.join();
    if (!ready) return kNone;
    if (!bad && !failed) return kDone;
    api.drain();
    return kFailed;
  }

  // the memory and every event, or nothing
  bool make(Api& api) {
    if (mem_) return true;
    char* m = nullptr;
    if (!api.pinned(&m, kSlots * kChunk)) return false;
    for (int k = 0; k < kSlots; ++k)
      if (!api.make(&ev_[k])) {
        while (k-- > 0) api.destroy(ev_[k]);
        api.free_pinned(m);
        return false;
      }
    mem_ = m;
    return true;
  }
  void destroy(Api& api) {
    if (!mem_) return;
    for (auto& e : ev_) api.destroy(e);
    api.free_pinned(mem_);
    mem_ = nullptr;
  }

 private:
  char* mem_ = nullptr;
  typename Api::Event ev_[kSlots] = {};
};

}  // namespace onsas
