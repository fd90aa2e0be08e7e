// Workspaces by stream (host side).
//
// Calls of one context on several streams may be in flight at once, so each
// stream that needs a workspace has its own, of at most kSlots. A further
// stream takes over the one used longest ago and waits for its last call on
// the device, by an event; nothing here waits on the host. (Events are recorded
// from the first take-over on, so that programs of up to kSlots streams record
// none; a workspace last used before that is kept aside instead.)
//
// Calls captured into a graph never share a workspace with calls that are not:
// the graph writes it at every replay, whenever that is. A capturing stream has
// buffers of its own, sized in powers of two, which live as long as the pool.
// It gets one only when the pool already holds one of that size or larger: the
// first call of a shape is made outside a capture.
//
// Rt: the runtime. Stream and Event (handles, null when zero), each function
// true on success:
//   alloc(void** p, size_t bytes)   allowed while a stream is being captured
//   release(void* p)
//   create(Event* e), destroy(Event e), record(Event e, Stream s), wait(Stream s, Event e)

#pragma once

#include <stddef.h>
#include <stdint.h>

#include <vector>

namespace c4s {

// kFailed: a function of the runtime did (runtime() knows which way).
enum class PoolResult { kOk, kWouldGrow, kFailed };

template <class Rt>
class StreamPool {
 public:
  using Stream = typename Rt::Stream;
  using Event = typename Rt::Event;
  static constexpr int kSlots = 8;

  Rt& runtime() { return rt_; }

  // A workspace of at least `need` bytes for a call about to be queued on `s`.
  PoolResult take(Stream s, bool capturing, size_t need, void** out) {
    *out = nullptr;
    if (capturing) return take_captured(s, need, out);
    Slot* w = find(s);
    if (!w && n_ < kSlots) {
      w = &slot_[n_++];
      w->stream = s;
    } else if (!w) {
      w = &slot_[0];
      for (Slot& o : slot_)
        if (o.used < w->used) w = &o;
      if (w->recorded) {
        if (!rt_.wait(s, w->done)) return PoolResult::kFailed;
      } else if (w->p) {
        aside_.push_back(w->p);   // until the pool goes: its last call may still run
        w->p = nullptr;
        w->bytes = 0;
      }
      turnover_ = true;
      w->stream = s;
    }
    if (w->bytes < need) {
      if (w->p) {
        const bool ok = rt_.release(w->p);
        w->p = nullptr;
        w->bytes = 0;
        if (!ok) return PoolResult::kFailed;
      }
      if (!rt_.alloc(&w->p, need)) {
        w->p = nullptr;
        return PoolResult::kFailed;
      }
      w->bytes = need;
    }
    w->used = ++tick_;
    w->recorded = false;
    *out = w->p;
    return PoolResult::kOk;
  }

  // The call that took a workspace on `s` has been queued.
  void queued(Stream s, bool capturing) {
    if (!turnover_ || capturing) return;
    Slot* w = find(s);
    if (!w) return;
    if (!w->done && !rt_.create(&w->done)) return;
    w->recorded = rt_.record(w->done, s);
  }

  // Everything given back; the streams' work has ended.
  void clear() {
    for (Slot& w : slot_) {
      if (w.p) (void)rt_.release(w.p);
      if (w.done) (void)rt_.destroy(w.done);
      w = Slot();
    }
    for (const Captured& c : captured_) (void)rt_.release(c.p);
    for (void* p : aside_) (void)rt_.release(p);
    captured_.clear();
    aside_.clear();
    n_ = 0;
    turnover_ = false;
  }

 private:
  struct Slot {
    Stream stream{};
    void* p = nullptr;
    size_t bytes = 0;
    uint64_t used = 0;       // tick of its last call
    Event done{};
    bool recorded = false;   // `done` marks the end of its last call
  };
  struct Captured {
    Stream stream;
    void* p;
    size_t bytes;
  };

  Slot* find(Stream s) {
    for (int i = 0; i < n_; ++i)
      if (slot_[i].stream == s) return &slot_[i];
    return nullptr;
  }

  PoolResult take_captured(Stream s, size_t need, void** out) {
    size_t largest = 0;
    for (int i = 0; i < n_; ++i) largest = slot_[i].bytes > largest ? slot_[i].bytes : largest;
    for (const Captured& c : captured_) {
      if (c.stream == s && c.bytes >= need) {
        *out = c.p;
        return PoolResult::kOk;
      }
      largest = c.bytes > largest ? c.bytes : largest;
    }
    if (largest < need) return PoolResult::kWouldGrow;
    size_t bytes = 1;
    while (bytes < need) bytes <<= 1;
    void* p = nullptr;
    if (!rt_.alloc(&p, bytes)) return PoolResult::kFailed;
    captured_.push_back({s, p, bytes});
    *out = p;
    return PoolResult::kOk;
  }

  Rt rt_;
  Slot slot_[kSlots];
  int n_ = 0;
  uint64_t tick_ = 0;
  bool turnover_ = false;
  std::vector<Captured> captured_;
  std::vector<void*> aside_;
};

}  // namespace c4s
