// The device's large workspace (urbilateria_amd/csrc/urb_large_work.hpp) over a stand-in for the
// GPU runtime: host memory with a limit, streams and events as counters of what they are ordered
// after.  Checks its bounds, that memory comes back, and that whatever threads and streams do, each
// use is ordered after the one before it and no memory is freed under a use.
#include "../../urbilateria_amd/csrc/urb_large_work.hpp"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <thread>
#include <vector>

#define CHECK(c)                                              \
  do {                                                        \
    if (!(c)) {                                               \
      std::printf("line %d: %s\n", __LINE__, #c);             \
      std::exit(1);                                           \
    }                                                         \
  } while (0)

struct FakeStream {
  long after = 0;  // the last use this stream's next work is ordered behind
  bool captured = false;
};
static FakeStream default_stream;  // the null handle's
static FakeStream& stream(FakeStream* s) { return s ? *s : default_stream; }

// All of it is called under LargeWork's mutex.
struct FakeGpu {
  using Stream = FakeStream*;
  using Event = long*;
  using Error = int;
  static constexpr Error kOk = 0, kNoMemory = 2;
  static constexpr size_t kBroken = 77;  // an allocation that fails for another reason
  static inline size_t capacity = 0, held = 0;
  static inline int allocations = 0, events = 0, device_syncs = 0, records = 0;
  static inline long last_use = 0, waited = 0;  // uses so far; the last one the host waited for
  static inline bool record_fails = false, sync_fails = false;
  static inline std::map<void*, size_t> sizes;
  static size_t free_bytes() { return capacity - held; }
  static Error alloc(void** p, size_t bytes) {
    if (bytes == kBroken) return 1;
    if (bytes > free_bytes()) return kNoMemory;
    *p = std::malloc(bytes);
    sizes[*p] = bytes;
    held += bytes;
    ++allocations;
    return kOk;
  }
  static void free(void* p) {
    CHECK(waited == last_use);  // nothing may still run on it
    held -= sizes.at(p);
    sizes.erase(p);
    std::free(p);
  }
  static bool create_event(Event* e) { *e = new long(0); ++events; return true; }
  static void destroy_event(Event e) { delete e; --events; }
  static bool record(Event e, Stream s) {
    if (record_fails) return false;
    *e = stream(s).after;
    ++records;
    return true;
  }
  static bool wait(Stream s, Event e) {
    if (stream(s).after < *e) stream(s).after = *e;
    return true;
  }
  static void wait_host(Event e) { waited = *e; }
  static bool sync() {
    if (sync_fails) return false;
    waited = last_use;
    ++device_syncs;
    return true;
  }
  static bool capturing(Stream s) { return stream(s).captured; }
};
using Work = urb::LargeWork<FakeGpu>;

// One use: it must come after the one before it (or the host waited for that one).
static bool use(Work& w, FakeStream* handle, size_t bytes, bool whole = true) {
  FakeStream& s = stream(handle);
  return w.run(handle, bytes, [&](void* base) {
    CHECK(s.after == FakeGpu::last_use || FakeGpu::waited == FakeGpu::last_use);
    std::memset(base, 1, bytes);
    s.after = ++FakeGpu::last_use;
    return whole;
  });
}

int main() {
  {
    Work w;
    FakeStream a, b;
    FakeGpu::capacity = 8000;
    CHECK(!use(w, &a, 1) && !w.release());
    w.attach(1001);                        // more than an eighth of what is free
    CHECK(FakeGpu::held == 0 && !use(w, &a, 1001));
    w.attach(500);
    CHECK(FakeGpu::held == 500 && use(w, &a, 500) && use(w, &b, 300) && use(w, &a, 500));
    CHECK(!use(w, &a, 501));                // not what this context needs
    w.attach(400);                         // fits what is there
    CHECK(FakeGpu::held == 500 && FakeGpu::allocations == 1);
    w.attach(1000);                        // the larger one takes its place: never two
    CHECK(FakeGpu::held == 1000 && use(w, &b, 1000));
    w.attach(1001);                        // too large: the one that is there stays
    CHECK(FakeGpu::held == 1000 && use(w, &a, 1000));
    b.captured = true;                     // a graph's call keeps off it
    CHECK(!use(w, &b, 10));
    CHECK(FakeGpu::device_syncs == 0);     // events alone so far
    CHECK(use(w, &a, 1000, false) && use(w, &a, 1000));  // stopped half-way: the next waits
    CHECK(FakeGpu::device_syncs == 1);
    FakeGpu::record_fails = true;
    CHECK(use(w, &a, 1000));
    FakeGpu::record_fails = false;
    FakeGpu::sync_fails = true;            // nothing orders the next call: it keeps off
    CHECK(!use(w, &a, 1000));
    FakeGpu::sync_fails = false;
    CHECK(use(w, &a, 1000) && FakeGpu::device_syncs == 2);
    CHECK(w.release() && FakeGpu::held == 0 && !use(w, &a, 10) && !w.release());
    w.attach(200);
    CHECK(FakeGpu::held == 200 && use(w, &a, 200));
    for (int i = 0; i < 5; ++i) w.detach();
    CHECK(FakeGpu::held == 200);
    w.detach();                            // the last of six contexts
    CHECK(FakeGpu::held == 0 && FakeGpu::events == 0);
  }
  {
    // a context's memory comes first: the region is given back before there is none, and only then
    Work w;
    FakeStream a;
    void *p = nullptr, *q = nullptr;
    w.attach(1000);
    CHECK(use(w, &a, 1000) && w.allocate(&p, 7000) == FakeGpu::kOk && FakeGpu::held == 8000);
    CHECK(w.allocate(&q, FakeGpu::kBroken) == 1 && FakeGpu::held == 8000);
    CHECK(w.allocate(&q, 600) == FakeGpu::kOk && FakeGpu::held == 7600 && !use(w, &a, 10));
    void* r = nullptr;
    CHECK(w.allocate(&r, 401) == FakeGpu::kNoMemory);
    w.attach(50);                          // an eighth of 400
    CHECK(FakeGpu::held == 7650 && use(w, &a, 50));
    FakeGpu::waited = FakeGpu::last_use;   // (free checks it for the region)
    FakeGpu::free(p);
    FakeGpu::free(q);
    w.detach();
    w.detach();
    CHECK(FakeGpu::held == 0 && FakeGpu::events == 0);
  }
  {
    // the default stream: an event only when another stream follows
    Work w;
    FakeStream a;
    FakeGpu::device_syncs = FakeGpu::records = 0;
    w.attach(500);
    for (int i = 0; i < 3; ++i) CHECK(use(w, nullptr, 500));
    CHECK(FakeGpu::records == 0 && use(w, &a, 500) && FakeGpu::records == 2);
    CHECK(use(w, nullptr, 500) && use(w, nullptr, 500) && FakeGpu::records == 2);
    FakeGpu::record_fails = true;
    CHECK(FakeGpu::device_syncs == 0 && use(w, &a, 500) && FakeGpu::device_syncs == 1);
    FakeGpu::record_fails = false;
    CHECK(use(w, nullptr, 500));
    w.detach();
    CHECK(FakeGpu::held == 0 && FakeGpu::events == 0);
  }
  {
    Work w;
    FakeGpu::capacity = 1 << 20;
    std::atomic<int> ran{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
      threads.emplace_back([&, t] {
        FakeStream own;
        unsigned r = 1u + (unsigned)t;
        const size_t bytes = 100 + 50 * (size_t)t;
        w.attach(bytes);
        for (int i = 0; i < 2000; ++i) {
          r = r * 1664525u + 1013904223u;
          switch (r >> 28) {
            case 0: w.release(); break;
            case 1: w.detach(); w.attach(bytes); break;
            case 2: w.attach(600); w.detach(); break;
            default: ran += use(w, (r >> 20) & 1 ? &own : nullptr, bytes) ? 1 : 0;
          }
        }
        w.detach();
      });
    for (auto& th : threads) th.join();
    CHECK(FakeGpu::held == 0 && FakeGpu::events == 0 && ran > 0);
  }
  std::printf("workspace driver ok\n");
  return 0;
}
