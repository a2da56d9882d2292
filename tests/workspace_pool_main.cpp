// The pool of device scratch (simplang_amd/runtime/workspace.h) over a memory
// that counts: run by test_workspace_pool.py.
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

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

struct Event {  // of a stream: kernels, and frees (which follow a drain)
  char what;
  void *buf;
  int who;
};
struct State {
  std::mutex mu;
  std::vector<Event> stream;
  bool capturing = false;
  size_t limit = ~size_t(0), held = 0, syncs = 0, allocs = 0;
  std::map<void *, size_t> live;
};
struct FakeMem {
  using Stream = int;
  State *s;
  bool capturing(int) const { return s->capturing; }
  void *alloc(size_t n) const {
    std::lock_guard<std::mutex> lk(s->mu);
    if (s->held + n > s->limit) return nullptr;
    void *p = (void *)(4096 * ++s->allocs);  // an address of its own, never read
    s->live[p] = n;
    s->held += n;
    return p;
  }
  bool sync(int) const {
    std::lock_guard<std::mutex> lk(s->mu);
    return ++s->syncs, true;
  }
  bool free(void *p) const {
    std::lock_guard<std::mutex> lk(s->mu);
    s->stream.push_back({'f', p, -1});
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
  Pool::Lease lease;
  CHECK(p.get(Pool::Key{0, stream, nullptr, slot}, bytes, &ptr, lease) == want);
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

// Threads on one stream: each call's launches stay together, and no buffer is
// freed between a lookup and the launches that use it.
void threads_share_a_stream() {
  State s;
  Pool p(FakeMem{&s});
  auto enqueue = [&](char what, void *buf, int who) {
    std::lock_guard<std::mutex> lk(s.mu);
    s.stream.push_back({what, buf, who});
  };
  std::vector<std::thread> ts;
  for (int t = 0; t < 4; t++)
    ts.emplace_back([&, t] {
      for (int i = 0; i < 500; i++) {
        void *buf = nullptr;
        Pool::Lease lease;
        CHECK(p.get(Pool::Key{0, 0, nullptr, 5}, (size_t)(1 + (7 * i + t) % 500) * (MB / 8), &buf,
                    lease) == WsStatus::kOk);
        enqueue('w', buf, t);
        std::this_thread::yield();
        enqueue('r', buf, t);
      }
    });
  for (auto &t : ts) t.join();
  std::map<void *, int> holds;  // buffer -> whose data, -1 once freed
  for (const Event &e : s.stream) {
    if (e.what == 'f') holds[e.buf] = -1;
    CHECK(e.what != 'w' || !holds.count(e.buf) || holds[e.buf] != -1);
    if (e.what == 'w') holds[e.buf] = e.who;
    CHECK(e.what != 'r' || holds[e.buf] == e.who);
  }
  CHECK(s.stream.size() > 4000 && s.syncs > 0);
}

int main() {
  graphs_keep_their_buffers();
  capture_needs_a_warm_up();
  what_stays_behind_is_bounded();
  no_memory();
  threads_share_a_stream();
  std::puts("ok");
}
