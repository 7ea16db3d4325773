// urb_large_work.hpp -- one device's workspace for layer calls beyond a context's own chunk.
//
// A call is fastest as one chunk, because every chunk reads each of its experts' weights, and one
// chunk of 4096 tokens holds 1.4 GB of buffers (7168 wide, top-8).  A model has a context per layer
// but runs its layers one after another, so the contexts of a device share one such region instead
// of each keeping it beside its weights: a context's own workspace stays at kOwnChunkTokens.
//
//  * Bounded: one region per device, as large as its largest context asks for, taken at creation
//    and only while it is at most an eighth of the free memory.
//  * Given back: when the last context that could use it is destroyed, and as soon as a creation
//    runs out of memory (allocate), so it never takes the place of a layer's weights.  Calls then
//    run in chunks of their own workspace.
//  * Threads and streams: a mutex covers a call's launches, and each call is ordered after the
//    region's last one, whichever stream that ran on: by an event, but on the default stream only
//    once another stream follows (that stream is never destroyed, so the event can be recorded
//    then).  An event after every call costs the next one 6 us if it forks at once (1900 tokens,
//    256 BF16 experts of 2048 x 512 with a shared one: 550 -> 557 us).  Calls of this size fill the
//    GPU, so streams lose nothing by taking turns.
//  * A call under stream capture never uses it: a graph keeps its addresses and replays outside of
//    this order, so it gets the context's own workspace.
//
// Gpu: the runtime calls as static functions (HIP in urb_moe_host.cpp, a stand-in in the test).
#pragma once

#include <cstddef>
#include <mutex>

namespace urb {

template <class Gpu>
class LargeWork {
 public:
  using Stream = typename Gpu::Stream;

  // A context whose longest chunk takes `bytes`: grows the region where memory allows it.
  void attach(size_t bytes) {
    std::lock_guard<std::mutex> lock(m_);
    ++users_;
    if (bytes <= bytes_ || bytes > (Gpu::free_bytes() + bytes_) / 8) return;
    drop();
    void* p = nullptr;
    if (Gpu::alloc(&p, bytes) != Gpu::kOk) return;
    if (!Gpu::create_event(&done_)) {
      Gpu::free(p);
      return;
    }
    base_ = p;
    bytes_ = bytes;
  }

  void detach() {
    std::lock_guard<std::mutex> lock(m_);
    if (--users_ == 0) drop();
  }

  // Device memory for a context's own use: before there is none, the region's is given back.
  typename Gpu::Error allocate(void** p, size_t bytes) {
    const typename Gpu::Error e = Gpu::alloc(p, bytes);
    return e == Gpu::kNoMemory && release() ? Gpu::alloc(p, bytes) : e;
  }

  // Gives the region's memory back; whether there was any.
  bool release() {
    std::lock_guard<std::mutex> lock(m_);
    const bool any = base_ != nullptr;
    drop();
    return any;
  }

  // Calls enqueue(base) with the region, ordered on `s` after its last use, when there are `bytes`
  // of it and `s` is not being captured; whether it did.  `enqueue` puts all its work on `s` (or
  // joins it there) and returns false if it stopped half-way.
  template <class F>
  bool run(Stream s, size_t bytes, F enqueue) {
    std::lock_guard<std::mutex> lock(m_);
    if (!base_ || bytes_ < bytes || Gpu::capturing(s) || !follow(s)) return false;
    const bool whole = enqueue(base_);
    if (whole && s == Stream{}) last_ = kDefaultStream;
    else last_ = whole && Gpu::record(done_, s) ? kEvent : kAnywhere;
    return true;
  }

 private:
  // What the region's last call is behind: nothing left to wait for, the event `done_`, the end of
  // the default stream, or no one place.
  enum Last { kNothing, kEvent, kDefaultStream, kAnywhere };

  // Orders `s` after the last call.
  bool follow(Stream s) {
    if (last_ == kDefaultStream) {
      if (s == Stream{}) return true;
      last_ = Gpu::record(done_, Stream{}) ? kEvent : kAnywhere;
    }
    if (last_ == kAnywhere) {
      if (!Gpu::sync()) return false;
      last_ = kNothing;
    }
    return last_ == kNothing || Gpu::wait(s, done_);
  }

  void drop() {
    if (!base_) return;
    if (last_ == kEvent) Gpu::wait_host(done_);
    else if (last_ != kNothing) (void)Gpu::sync();
    Gpu::destroy_event(done_);
    Gpu::free(base_);
    base_ = nullptr;
    bytes_ = 0;
    last_ = kNothing;
  }

  std::mutex m_;
  void* base_ = nullptr;
  size_t bytes_ = 0;
  int users_ = 0;
  typename Gpu::Event done_{};
  Last last_ = kNothing;
};

}  // namespace urb
