// BlockCache's stream-ordered blocks (csrc/device_cache.h) over a malloc
// backend: only alloc_ordered hands a release_ordered block out before
// settle, a failed wait keeps it apart, trim returns it, counts stay whole, and
// holds (which lets a kernel read a caller's range) knows where blocks end.
#include <cstdio>
#include <cstdlib>

#include "device_cache.h"

using namespace tt;

static int g_failures = 0;
#define CHECK(cond) \
  do { \
    if (!(cond)) { std::fprintf(stderr, "line %d: %s\n", __LINE__, #cond); ++g_failures; } \
  } while (0)

struct Backend {
  int releases = 0;
  int alloc(size_t bytes, void** p) { return (*p = std::malloc(bytes)) ? 0 : 4; }
  void release(void* p) { std::free(p), ++releases; }
};

static void holds_checks() {
  Backend be;
  BlockCache<Backend> bc(be);
  char host[64], *a, *b;
  CHECK(!bc.holds(host, 1));
  CHECK(bc.alloc(4096, (void**)&a) == 0 && bc.alloc_ordered(1000, (void**)&b) == 0);  // b: a class of 1024
  for (char* p : {a, b}) {
    const size_t n = p == a ? 4096 : 1024;
    CHECK(bc.holds(p, n) && bc.holds(p + 16, n - 16) && bc.holds(p + n - 1, 1) && bc.holds(p, 0));
    CHECK(!bc.holds(p, n + 1) && !bc.holds(p + 16, n - 15) && !bc.holds(p + n, 1));
    CHECK(!bc.holds(p, ~size_t(0)) && !bc.holds(p + 16, ~size_t(0)));
  }
  CHECK(!bc.holds(nullptr, 1) && !bc.holds(host, 1));
  CHECK(bc.release(a) && !bc.holds(a, 1) && bc.holds(b, 1));  // cached, not live
  CHECK(bc.release_ordered(b) && !bc.holds(b, 1));
  bc.trim();
}

// Another thread's calls while settle waits (made from inside the wait).
static void settle_window_checks() {
  Backend be;
  BlockCache<Backend> bc(be);
  void *a, *b, *c = nullptr;
  size_t used, cached;
  // a trim returns the waiting blocks too, and the counts stay whole
  CHECK(bc.alloc_ordered(4096, &a) == 0 && bc.release_ordered(a));
  CHECK(bc.settle([&] { return bc.trim(), 0; }) == 0);
  CHECK(be.releases == 1);
  CHECK(bc.alloc(4096, &a) == 0 && bc.release(a) && bc.alloc(4096, &a) == 0);
  bc.stats(&used, &cached);
  CHECK(used == 4096 && cached == 0);
  // one taken meanwhile is gone; one released meanwhile is not covered by the wait
  CHECK(bc.alloc_ordered(8192, &b) == 0 && bc.alloc_ordered(8192, &c) == 0);
  CHECK(bc.release_ordered(b));
  void* d = nullptr;
  CHECK(bc.settle([&] {
    CHECK(bc.alloc_ordered(8192, &d) == 0 && d == b);
    CHECK(bc.release_ordered(c));
    return 0;
  }) == 0);
  bc.stats(&used, &cached);
  CHECK(used == 4096 + 8192 && cached == 8192);
  CHECK(bc.wants_settle(8192));  // c waits still
  CHECK(bc.release(a) && bc.release(d));
  bc.trim();
  bc.stats(&used, &cached);
  CHECK(used == 0 && cached == 0);
}

int main() {
  holds_checks();
  settle_window_checks();
  Backend be;
  BlockCache<Backend> bc(be);
  void *a = nullptr, *b = nullptr, *c = nullptr;
  CHECK(bc.alloc_ordered(4096, &a) == 0);
  CHECK(!bc.wants_settle(4096));
  CHECK(bc.release_ordered(a) && !bc.release_ordered(a) && !bc.release(a));
  CHECK(bc.wants_settle(4096) && !bc.wants_settle(1 << 20));
  CHECK(bc.alloc(4096, &b) == 0 && b != a);          // never before settle
  CHECK(bc.settle([] { return 5; }) == 5);           // a failed wait
  CHECK(bc.alloc(4096, &c) == 0 && c != a);
  CHECK(bc.release(c));
  CHECK(!bc.wants_settle(4096));                     // an ordinary block serves it
  CHECK(bc.alloc_ordered(4096, &c) == 0 && c == a);  // the ordered block first
  CHECK(bc.release_ordered(c));
  CHECK(bc.settle([] { return 0; }) == 0);
  size_t used = 0, cached = 0;
  bc.stats(&used, &cached);
  CHECK(used == 4096 && cached == 8192);
  CHECK(bc.alloc(4096, &a) == 0 && bc.alloc(4096, &c) == 0);  // both cached blocks
  bc.stats(&used, &cached);
  CHECK(used == 3 * 4096 && cached == 0);
  CHECK(bc.release_ordered(a) && bc.release(b) && bc.release_ordered(c));
  bc.trim();
  CHECK(be.releases == 3);
  bc.stats(&used, &cached);
  CHECK(used == 0 && cached == 0);
  if (!g_failures) std::puts("ordered checks passed");
  return g_failures ? 1 : 0;
}
