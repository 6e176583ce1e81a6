// The block cache over a driver of its own (no GPU): memory that queued work
// may use is not handed out before a wait for the device has succeeded.
#include <cstdio>
#include <cstdlib>
#include <set>
#include <vector>

#include "drx_blocks.hpp"

static int failures = 0;
#define CHECK(c)                                                     \
  do {                                                               \
    if (!(c)) {                                                      \
      std::printf("line %d: %s\n", __LINE__, #c);                    \
      failures++;                                                    \
    }                                                                \
  } while (0)

struct Fake {
  static constexpr int kOutOfMemory = 2;
  static inline std::set<void *> live;
  static inline size_t room = SIZE_MAX, used = 0;
  static inline std::map<void *, size_t> bytes;
  static inline bool may_wait = true, may_free = true;
  static inline int waits = 0;
  static int alloc(void **p, size_t n) {
    if (n > room - used) return kOutOfMemory;
    *p = std::malloc(64);
    used += n;
    live.insert(*p);
    bytes[*p] = n;
    return 0;
  }
  static bool free(void *p) {
    if (!may_free) return false;
    used -= bytes[p];
    live.erase(p);
    std::free(p);
    return true;
  }
  static bool wait() {
    waits++;
    return may_wait;
  }
};
constexpr size_t MB = size_t(1) << 20;
using Cache = drx::BlockCache<Fake, 8 * MB>;

static void *take(Cache &c, size_t n) {
  void *p = nullptr;
  return c.take(n, &p) == 0 ? p : nullptr;
}

int main() {
  {  // a refused wait: the blocks serve nobody, and come back after the next one
    Cache c;
    void *a = take(c, MB), *b = take(c, 2 * MB);
    Fake::may_wait = false;
    c.retire(std::initializer_list<void *>{a, b, nullptr});
    CHECK(c.kept() == 0);
    void *n1 = take(c, MB), *n2 = take(c, 2 * MB);
    CHECK(n1 != a && n1 != b && n2 != a && n2 != b);
    CHECK(Fake::live.count(a) && Fake::live.count(b));
    CHECK(!c.release());
    CHECK(Fake::live.count(a) && Fake::live.count(b));
    c.retire(std::initializer_list<void *>{n1});
    CHECK(c.kept() == 0);
    Fake::may_wait = true;
    CHECK(c.settle());
    CHECK(c.kept() == 4 * MB);
    void *m = take(c, 2 * MB);
    CHECK(m == b);
    CHECK(c.release() && c.kept() == 0);
    c.give(n2);
    c.give(m);
    c.release();
  }
  CHECK(Fake::live.empty());
  {  // no wait without a retired block; one per retirement; give takes none
    Cache c;
    Fake::waits = 0;
    void *a = take(c, 10);
    c.give(a);
    CHECK(take(c, 4096) == a && Fake::waits == 0);
    c.retire(std::initializer_list<void *>{a});
    CHECK(Fake::waits == 1 && c.kept() == 4096);
    c.retire(std::initializer_list<void *>{nullptr});
    CHECK(Fake::waits == 1);
    c.release();
  }
  CHECK(Fake::live.empty());
  {  // at most 8 MB kept, oldest given back first; a block far too large is not used
    Cache c;
    std::vector<void *> v;
    for (int i = 0; i < 10; i++) v.push_back(take(c, MB));
    for (void *p : v) c.give(p);
    CHECK(c.kept() == 8 * MB && !Fake::live.count(v[0]) && Fake::live.count(v[9]));
    void *s = take(c, 4096);
    CHECK(c.kept() == 8 * MB);
    c.give(s);
    // a driver that refuses frees keeps them (and the loop ends)
    Fake::may_free = false;
    CHECK(!c.release());
    void *t = take(c, 16 * MB);
    c.give(t);
    CHECK(c.kept() > 8 * MB);
    Fake::may_free = true;
    CHECK(c.release() && c.kept() == 0);
  }
  CHECK(Fake::live.empty());
  {  // out of memory: kept and settled blocks go back, then the allocation passes
    Cache c;
    Fake::room = 6 * MB;
    void *a = take(c, 3 * MB), *b = take(c, 2 * MB);
    c.give(a);
    CHECK(take(c, 5 * MB) == nullptr);  // b is in use
    Fake::may_wait = false;
    c.retire(std::initializer_list<void *>{b});
    CHECK(take(c, 5 * MB) == nullptr);  // b may still be read
    Fake::may_wait = true;
    void *d = take(c, 5 * MB);
    CHECK(d != nullptr);
    c.give(d);
    c.release();
    Fake::room = SIZE_MAX;
  }
  CHECK(Fake::live.empty());
  std::printf("%d failures\n", failures);
  return failures != 0;
}
