// The pool of device scratch (simplang_amd/runtime/workspace.h) over a memory
// that counts: run by test_workspace_pool.py.
#include <cstdio>
#include <cstdlib>
#include <set>

#include "workspace.h"

using namespace simp;

#define CHECK(c)                                            \
  do {                                                      \
    if (!(c)) {                                             \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);   \
      std::exit(1);                                         \
    }                                                       \
  } while (0)

constexpr size_t MB = size_t(1) << 20;

struct State {
  bool capturing = false;
  size_t limit = ~size_t(0), held = 0, syncs = 0, allocs = 0;
  std::map<void *, size_t> live;
};
struct FakeMem {
  using Stream = int;
  State *s;
  bool capturing(int) const { return s->capturing; }
  void *alloc(size_t n) const {
    if (s->held + n > s->limit) return nullptr;
    void *p = (void *)(4096 * ++s->allocs);  // an address of its own, never read
    s->live[p] = n;
    s->held += n;
    return p;
  }
  bool sync(int) const { return ++s->syncs, true; }
  bool free(void *p) const {
    CHECK(s->live.count(p));
    s->held -= s->live[p];
    s->live.erase(p);
    return true;
  }
};
using Pool = WsPool<FakeMem>;

void *get(Pool &p, State &s, bool capturing, size_t bytes, WsStatus want = WsStatus::kOk, int stream = 0,
          int slot = 3) {
  s.capturing = capturing;
  void *ptr = nullptr;
  CHECK(p.get(Pool::Key{0, stream, slot}, bytes, &ptr) == want);
  CHECK(want != WsStatus::kOk || s.live.at(ptr) >= bytes);
  return ptr;
}

// What a graph was recorded with stays allocated, and no eager call gets it.
void graphs_keep_their_buffers() {
  State s;
  Pool p(FakeMem{&s});
  void *e = get(p, s, false, 2 * MB);
  void *g = get(p, s, true, 2 * MB);
  CHECK(g == e);                               // the warm-up's
  void *e2 = get(p, s, false, 2 * MB);
  CHECK(e2 != g);
  get(p, s, false, 8 * MB);                    // grows: frees e2, not g
  CHECK(s.live.count(g) && !s.live.count(e2) && s.syncs == 1);
  CHECK(get(p, s, true, 1 * MB) == g);         // a second graph shares it
  void *g2 = get(p, s, true, 8 * MB);          // a larger one
  CHECK(g2 != g && s.live.count(g));
  CHECK(get(p, s, true, 2 * MB) == g2);
}

// A capture without a warm-up of its size is refused, as it cannot allocate.
void capture_needs_a_warm_up() {
  State s;
  Pool p(FakeMem{&s});
  get(p, s, true, 2 * MB, WsStatus::kCapturing);
  get(p, s, false, 2 * MB);
  get(p, s, true, 3 * MB, WsStatus::kCapturing);
  get(p, s, true, 2 * MB, WsStatus::kCapturing, 1);     // another stream
  get(p, s, true, 2 * MB, WsStatus::kCapturing, 0, 2);  // another slot
  get(p, s, true, 2 * MB);
  CHECK(s.held == 2 * MB);
}

// Every larger capture leaves a buffer behind: together less than the last.
void what_stays_behind_is_bounded() {
  State s;
  Pool p(FakeMem{&s});
  size_t n = 2 * MB;
  for (int i = 0; i < 200; i++, n += MB / 4) {
    get(p, s, false, n);
    get(p, s, true, n);
  }
  CHECK(s.held <= 6 * n);  // graphs: at most 2 n and what is behind it; eager: at most n
}

// No memory: reported, and the pool goes on with what it has.
void no_memory() {
  State s;
  s.limit = 5 * MB;
  Pool p(FakeMem{&s});
  get(p, s, false, 2 * MB);
  get(p, s, false, 6 * MB, WsStatus::kNoMemory);
  get(p, s, false, 2 * MB);
  get(p, s, true, 2 * MB);
  get(p, s, false, 3 * MB);  // twice the graphs' does not fit, 3 MB does
  CHECK(s.held == 5 * MB);
}

int main() {
  graphs_keep_their_buffers();
  capture_needs_a_warm_up();
  what_stays_behind_is_bounded();
  no_memory();
  std::puts("ok");
}
