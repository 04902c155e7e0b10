// The ring of the large downloads (onsas.jl_amd/csrc/copy_ring.hpp) on a device made of a
// thread: every value in its place, slots reused only when they are empty, and what is
// left when pinned memory, an event or a copy is refused.
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <functional>
#include <mutex>
#include <set>

#include "copy_ring.hpp"

using namespace onsas;

#define CHECK(c)                                           \
  do {                                                     \
    if (!(c)) {                                            \
      std::fprintf(stderr, "line %d: %s\n", __LINE__, #c); \
      std::exit(1);                                        \
    }                                                      \
  } while (0)

// A stream that one thread works through; an event is done when its last record has run.
struct Device {
  using Event = int;
  std::mutex mu;
  std::condition_variable cv;
  std::deque<std::function<void()>> jobs;
  bool busy = false, stop = false;
  std::vector<int64_t> asked, done;  // per event: records queued, run
  std::set<Event> live;
  int blocks = 0;                    // pinned allocations not given back
  // what is refused: the n-th call of its kind from now (0: none)
  int no_pinned = 0, no_event = 0, no_copy = 0, no_wait = 0;
  std::thread t{[this] {
    std::unique_lock<std::mutex> l(mu);
    for (;;) {
      cv.wait(l, [this] { return stop || !jobs.empty(); });
      if (jobs.empty()) return;
      auto j = std::move(jobs.front());
      jobs.pop_front();
      busy = true;
      l.unlock();
      j();
      l.lock();
      busy = false;
      cv.notify_all();
    }
  }};
  ~Device() {
    {
      std::lock_guard<std::mutex> l(mu);
      stop = true;
    }
    cv.notify_all();
    t.join();
  }
  static bool refuse(int& n) { return n > 0 && --n == 0; }
  void put(std::function<void()> f) {
    std::lock_guard<std::mutex> l(mu);
    jobs.push_back(std::move(f));
    cv.notify_all();
  }
  bool pinned(char** p, size_t n) {
    if (refuse(no_pinned)) return false;
    *p = new char[n];
    ++blocks;
    return true;
  }
  void free_pinned(char* p) {
    delete[] p;
    --blocks;
  }
  bool make(Event* e) {
    if (refuse(no_event)) return false;
    std::lock_guard<std::mutex> l(mu);
    *e = (int)asked.size();
    asked.push_back(0);
    done.push_back(0);
    live.insert(*e);
    return true;
  }
  void destroy(Event e) {
    std::lock_guard<std::mutex> l(mu);
    CHECK(live.erase(e) == 1);
  }
  bool queue(char* pin, const void* src, size_t n) {
    if (refuse(no_copy)) return false;
    put([=] { std::memcpy(pin, src, n); });
    return true;
  }
  bool record(Event e) {
    {
      std::lock_guard<std::mutex> l(mu);
      CHECK(live.count(e));
      ++asked[e];
    }
    put([this, e] {
      std::lock_guard<std::mutex> l(mu);
      ++done[e];
    });
    return true;
  }
  bool wait(Event e) {
    std::unique_lock<std::mutex> l(mu);
    if (refuse(no_wait)) return false;
    CHECK(live.count(e));
    const int64_t n = asked[e];
    cv.wait(l, [&] { return done[e] >= n; });
    return true;
  }
  void drain() {
    std::unique_lock<std::mutex> l(mu);
    cv.wait(l, [this] { return jobs.empty() && !busy; });
  }
};

using Ring = CopyRing<Device, 4096>;

struct Arrays {
  std::vector<std::vector<unsigned char>> src, dst;
  std::vector<CopyPart> parts;
  explicit Arrays(const std::vector<size_t>& bytes) {
    unsigned x = 1;
    for (size_t n : bytes) {
      src.emplace_back(n);
      dst.emplace_back(n + 1, 0xee);  // and a byte that stays
      for (auto& c : src.back()) c = (unsigned char)((x = x * 1664525u + 1013904223u) >> 24);
    }
    for (size_t i = 0; i < bytes.size(); ++i) parts.push_back({dst[i].data(), src[i].data(), bytes[i]});
  }
  bool in_place() const {
    for (size_t i = 0; i < src.size(); ++i)
      if (!std::equal(src[i].begin(), src[i].end(), dst[i].begin()) || dst[i].back() != 0xee)
        return false;
    return true;
  }
};

int main() {
  const size_t C = Ring::kChunk;
  const std::vector<std::vector<size_t>> sizes = {
      {1}, {C}, {C - 1, 1}, {C + 1, 7}, {3 * C, 0, 2 * C + 5}, {8 * C}, {9 * C - 3, 11}, {20 * C + 17}};
  {  // whole copies, the ring kept from one to the next
    Device d;
    Ring ring;
    for (int round = 0; round < 2; ++round)
      for (const auto& s : sizes) {
        Arrays a(s);
        CHECK(ring.copy(d, a.parts) == Ring::kDone && a.in_place());
      }
    CHECK(d.blocks == 1 && d.live.size() == 8);
    ring.destroy(d);
    CHECK(d.blocks == 0 && d.live.empty());
  }
  // refused pinned memory or events: nothing queued, nothing kept, and the next call has
  // another try
  for (int n = 0; n <= 8; ++n) {
    Device d;
    Ring ring;
    Arrays a({3 * C + 9});
    (n == 0 ? d.no_pinned : d.no_event) = n == 0 ? 1 : n;
    CHECK(ring.copy(d, a.parts) == Ring::kNone);
    CHECK(d.blocks == 0 && d.live.empty() && d.jobs.empty());
    CHECK(ring.copy(d, a.parts) == Ring::kDone && a.in_place());
    ring.destroy(d);
    CHECK(d.blocks == 0 && d.live.empty());
  }
  // a copy or a wait that fails, at any place: the call ends and says so, the stream is
  // idle, and the ring is good for the next one
  for (int n = 1; n <= 14; ++n)
    for (bool waits : {false, true}) {
      Device d;
      Ring ring;
      Arrays a({13 * C + 9});
      (waits ? d.no_wait : d.no_copy) = n;
      CHECK(ring.copy(d, a.parts) == Ring::kFailed);
      CHECK(d.jobs.empty() && !d.busy);
      Arrays b({5 * C});
      CHECK(ring.copy(d, b.parts) == Ring::kDone && b.in_place());
      ring.destroy(d);
      CHECK(d.blocks == 0 && d.live.empty());
    }
  std::puts("ok");
}
