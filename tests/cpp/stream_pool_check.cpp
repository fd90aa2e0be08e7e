// Workspaces by stream (csrc/c4s_pool.hpp) on a runtime that only keeps books:
// who may use which buffer, what a take-over waits for, and that everything is
// given back. Prints "0 failures".

#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include <vector>

#include "c4s_pool.hpp"

namespace {

struct Book {
  std::map<void*, size_t> live;                      // buffers not released
  std::map<int, std::pair<int, int>> event;          // event -> (stream, its calls when recorded)
  struct Wait { int stream, of, calls; };            // `stream` waits for the first `calls` calls of `of`
  std::vector<Wait> waits;
  std::map<void*, std::pair<int, int>> user;         // buffer -> its last user and that call's number
  std::map<int, int> calls;                          // calls queued on a stream
  int events = 0, records = 0, fail_alloc = 0;
} book;

struct FakeRt {
  using Stream = int;
  using Event = int;
  bool alloc(void** p, size_t n) {
    if (book.fail_alloc) return false;
    *p = std::malloc(1);
    book.live[*p] = n;
    return true;
  }
  bool release(void* p) {
    const bool ok = book.live.erase(p) == 1;
    book.user.erase(p);
    std::free(p);
    return ok;
  }
  bool create(int* e) { *e = ++book.events; return true; }
  bool destroy(int e) { book.event.erase(e); --book.events; return true; }
  bool record(int e, int s) {
    book.event[e] = {s, book.calls[s]};
    ++book.records;
    return true;
  }
  bool wait(int s, int e) { book.waits.push_back({s, book.event[e].first, book.event[e].second}); return true; }
};

using Pool = c4s::StreamPool<FakeRt>;
using c4s::PoolResult;
int failures = 0;
#define CHECK(c)                                                     \
  do {                                                               \
    if (!(c)) {                                                      \
      ++failures;                                                    \
      std::printf("line %d: %s\n", __LINE__, #c);                    \
    }                                                                \
  } while (0)

void* call(Pool& p, int s, size_t need, bool cap = false, PoolResult want = PoolResult::kOk) {
  void* w = nullptr;
  const size_t n_waits = book.waits.size();
  const PoolResult r = p.take(s, cap, need, &w);
  CHECK(r == want);
  CHECK((w != nullptr) == (r == PoolResult::kOk));
  if (w) CHECK(book.live.count(w) == 1 && book.live[w] >= need);
  if (!cap) ++book.calls[s];
  if (w && !cap) {
    const auto u = book.user.find(w);
    if (u != book.user.end() && u->second.first != s) {   // another stream's before: behind its last call
      CHECK(book.waits.size() == n_waits + 1);
      if (book.waits.size() > n_waits) {
        const Book::Wait& x = book.waits.back();
        CHECK(x.stream == s && x.of == u->second.first && x.calls >= u->second.second);
      }
    }
    book.user[w] = {s, book.calls[s]};
  }
  p.queued(s, cap);
  return w;
}

// A few streams: one buffer each, kept, no event, nothing waited for.
void few_streams() {
  Pool p;
  std::set<void*> seen;
  for (int s = 0; s < Pool::kSlots; ++s) {
    void* w = call(p, s, 100);
    CHECK(seen.insert(w).second);
    CHECK(call(p, s, 60) == w);
  }
  CHECK(book.records == 0 && book.waits.empty());
  p.clear();
  CHECK(book.live.empty());
}

// More streams than slots: the one used longest ago is taken over, its last
// call waited for by the event recorded behind it; a buffer whose last call has
// no event is not used again.
void many_streams() {
  book = Book();
  Pool p;
  std::vector<void*> first;
  for (int s = 0; s < Pool::kSlots; ++s) first.push_back(call(p, s, 100));
  void* w8 = call(p, Pool::kSlots, 100);
  CHECK(book.waits.empty());   // stream 0's call has no event: another buffer
  for (void* f : first) CHECK(f != w8);
  CHECK(book.live.count(first[0]) == 1);   // and that one is still there
  for (int round = 0; round < 50; ++round)
    for (int s = 100; s < 109; ++s) {
      void* w = call(p, s + (round % 3) * 9, 100);
      CHECK(w != first[0]);
    }
  CHECK(book.live.size() <= 2 * (size_t)Pool::kSlots);
  CHECK(!book.waits.empty());
  p.clear();
  CHECK(book.live.empty() && book.events == 0);
}

// Captured calls: buffers of their own, never handed to another call, whatever
// streams come and however the others grow; none without a call outside first.
void captures() {
  book = Book();
  Pool p;
  call(p, 1, 100, true, PoolResult::kWouldGrow);
  void* eager = call(p, 1, 100);
  call(p, 1, 101, true, PoolResult::kWouldGrow);
  void* cap1 = call(p, 1, 100, true);      // the same stream, captured
  void* cap2 = call(p, 2, 70, true);       // another, whose own call was never made
  CHECK(cap1 != eager && cap2 != eager && cap1 != cap2);
  CHECK(call(p, 1, 100) == eager);
  CHECK(call(p, 1, 90, true) == cap1);     // graphs of one stream share its buffer
  CHECK(call(p, 2, 70, true) == cap2);
  for (int round = 0; round < 4; ++round)
    for (int s = 0; s < 30; ++s) {
      void* w = call(p, s, 100 + 50 * round);
      CHECK(w != cap1 && w != cap2);
      CHECK(book.live.count(cap1) == 1 && book.live.count(cap2) == 1);
    }
  void* big = call(p, 1, 250, true);       // larger graphs: another, the old one stays
  CHECK(big != cap1 && book.live.count(cap1) == 1);
  CHECK(call(p, 1, 100, true) == cap1 && call(p, 1, 256, true, PoolResult::kOk) == big);
  // one captured size after another, rising: powers of two, so few buffers
  const size_t before = book.live.size();
  for (size_t n = 300; n < 3000; n += 7) {
    call(p, 1, n);
    call(p, 1, n, true);
  }
  CHECK(book.live.size() <= before + 5);
  p.clear();
  CHECK(book.live.empty());
}

void no_memory() {
  book = Book();
  Pool p;
  void* w = call(p, 1, 100);
  book.fail_alloc = 1;
  call(p, 2, 100, false, PoolResult::kFailed);
  call(p, 1, 200, false, PoolResult::kFailed);
  book.fail_alloc = 0;
  CHECK(book.live.count(w) == 0);
  call(p, 1, 200);
  call(p, 2, 100);
  p.clear();
  CHECK(book.live.empty());
}

}  // namespace

int main() {
  few_streams();
  many_streams();
  captures();
  no_memory();
  std::printf("%d failures\n", failures);
  return failures ? 1 : 0;
}
