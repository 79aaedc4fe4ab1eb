// The rules of csrc/scratch.h, with an allocator that counts.
#include "scratch.h"

#include <cstdio>
#include <cstdlib>
#include <set>
#include <thread>

using tinyoai::ScratchPool;

#define CHECK(x)                                           \
  do {                                                     \
    if (!(x)) {                                            \
      std::printf("line %d: %s\n", __LINE__, #x);          \
      std::exit(1);                                        \
    }                                                      \
  } while (0)

static std::set<void *> live;
static bool full = false;
static void *alloc(size_t bytes) {
  if (full || !bytes) return nullptr;
  void *p = std::malloc(16);
  live.insert(p);
  return p;
}
static void give(void *p) {
  CHECK(live.erase(p) == 1);  // once
  std::free(p);
}

int main() {
  const void *s[12];
  for (int i = 0; i < 12; i++) s[i] = reinterpret_cast<const void *>(uintptr_t(64 * (i + 1)));
  {
    ScratchPool p;
    // streams, and threads of one handle
    void *a = p.eager(s[0], 0, 100, alloc).ptr, *b = p.eager(s[1], 0, 100, alloc).ptr;
    void *t1 = p.eager(s[2], 1, 100, alloc).ptr, *t2 = p.eager(s[2], 2, 100, alloc).ptr;
    CHECK(std::set<void *>({a, b, t1, t2}).size() == 4);
    CHECK(p.eager(s[0], 0, 60, alloc).ptr == a && p.eager(s[2], 2, 100, alloc).ptr == t2);
    // a larger call keeps what enqueued work may use
    void *c = p.eager(s[0], 0, 120, alloc).ptr;
    CHECK(c != a && live.count(a) && p.eager(s[0], 0, 150, alloc).ptr == c);  // half as large again
    // captures: never a stream's buffer, nor another capture's or another stream's of the same one
    ScratchPool::Record *r1, *r2, *r3, *r4, *none;
    void *g1 = p.captured(7, s[0], 100, alloc, &r1), *g2 = p.captured(8, s[0], 100, alloc, &r2);
    void *g3 = p.captured(7, s[1], 100, alloc, &r3);
    CHECK(r1 && r2 && r3 && std::set<void *>({a, b, c, t1, t2, g1, g2, g3}).size() == 8);
    CHECK(p.captured(7, s[0], 80, alloc, &none) == g1 && !none);
    void *g4 = p.captured(7, s[0], 300, alloc, &r4);  // a larger call of the capture: the smaller one's stays
    CHECK(r4 && g4 != g1 && live.count(g1) && p.eager(s[0], 0, 100, alloc).ptr == c);
    // what a destroyed graph had goes to the next capture that it is large enough for
    const size_t count = live.size();
    std::thread(ScratchPool::release, r2).join();
    ScratchPool::Record *r5, *r6;
    void *g5 = p.captured(9, s[3], 200, alloc, &r5);
    CHECK(r5 && g5 != g2 && live.size() == count + 1);
    CHECK(p.captured(10, s[3], 100, alloc, &r6) == g2 && r6 && r6 != r2 && live.size() == count + 1);
    CHECK(p.captured(8, s[0], 100, alloc, &r2) != g2 && r2);  // an id again: not what its graph let go
    // out of memory: an error, and what is there stays
    full = true;
    CHECK(!p.captured(11, s[0], 100, alloc, &none) && !none);
    CHECK(!p.eager(s[0], 0, 1000, alloc).ptr && p.eager(s[0], 0, 100, alloc).ptr == c);
    full = false;
    // streams past the eighth share a buffer, and say so
    std::set<void *> own, shared;
    for (int i = 0; i < 12; i++) {
      const ScratchPool::Lease l = p.eager(s[i], 0, 100, alloc);
      (l.shared ? shared : own).insert(l.ptr);
      CHECK(p.eager(s[i], 0, 100, alloc).ptr == l.ptr);
    }
    CHECK(shared.size() == 1 && own.size() + 2 == ScratchPool::kStreams && !own.count(*shared.begin()));
    // graphs that outlive the pool
    ScratchPool::release(r1);
    p.clear(give);
    CHECK(live.empty());
    for (ScratchPool::Record *r : {r2, r3, r4, r5, r6}) ScratchPool::release(r);
  }
  std::printf("ok\n");
  return 0;
}
