// workspace.h -- the library's pool of device scratch, host code only (Mem
// stands for the HIP calls, so that the pool can be built and tested without
// them).
//
// One entry per (device, stream, slot) holds two buffers:
//   * `eager`, of the calls that are not captured.  It grows on demand; the old
//     buffer is freed once the stream has drained.
//   * `graph`, of the calls recorded into a graph.  A graph replays into the
//     address that it was recorded with for as long as the caller keeps it, so
//     this buffer is never freed, and no uncaptured call is given it: a replay
//     (on any stream, from any thread) then meets no eager call's data.  The
//     first captured call takes over the eager buffer that a warm-up call of
//     its size left; a captured call above it takes over a larger one, and the
//     old one stays behind for its graphs.  The eager buffer that such a call
//     needs is made twice as large as the graphs' one, so what stays behind
//     adds up to less than the buffer in use.
//
// A call that writes scratch with one launch and reads it with a later one holds
// a Lease from the lookup to its last launch: no other thread's call on the same
// stream then puts its launches in between, or frees the buffer by growing it.
// Leases nest in the order of the slots' users (a product that stages operands
// in one slot runs another product on them), never in a circle.
#pragma once

#include <algorithm>
#include <cstddef>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>

namespace simp {

enum class WsStatus {
  kOk,
  kCapturing,  // the stream is being captured and no buffer is large enough
  kNoMemory,
  kError,      // of Mem::sync or Mem::free
};

template <class Mem>
class WsPool {
 public:
  using Stream = typename Mem::Stream;
  // device, stream, the thread where the stream's handle names one per thread
  // (else null), slot
  using Key = std::tuple<int, Stream, const void *, int>;
  using Lease = std::unique_lock<std::mutex>;

  explicit WsPool(Mem mem = Mem()) : mem_(mem) {}

  // A buffer of at least `bytes` for the launches on the key's stream that the
  // caller makes while it holds `lease`.
  WsStatus get(const Key &key, size_t bytes, void **ptr, Lease &lease) {
    Entry &e = entry(key);
    lease = Lease(e.mu);
    const Stream st = std::get<1>(key);
    if (mem_.capturing(st)) {
      if (e.graph.bytes < bytes) {
        if (e.eager.bytes < bytes) return WsStatus::kCapturing;
        e.graph = e.eager;
        e.eager = Buf{};
      }
      *ptr = e.graph.ptr;
      return WsStatus::kOk;
    }
    if (e.eager.bytes < bytes) {
      if (e.eager.ptr) {
        if (!mem_.sync(st) || !mem_.free(e.eager.ptr)) return WsStatus::kError;
        e.eager = Buf{};
      }
      size_t want = std::max(bytes, kMin);
      void *p = nullptr;
      if (e.graph.bytes && bytes > e.graph.bytes) {
        const size_t twice = std::max(want, 2 * e.graph.bytes);
        if ((p = mem_.alloc(twice))) want = twice;
      }
      if (!p && !(p = mem_.alloc(want))) return WsStatus::kNoMemory;
      e.eager = Buf{p, want};
    }
    *ptr = e.eager.ptr;
    return WsStatus::kOk;
  }

 private:
  static constexpr size_t kMin = size_t(1) << 20;
  struct Buf {
    void *ptr = nullptr;
    size_t bytes = 0;
  };
  struct Entry {
    std::mutex mu;
    Buf eager, graph;
  };
  Entry &entry(const Key &key) {  // entries stay where they are
    std::lock_guard<std::mutex> lk(mu_);
    return entries_[key];
  }
  Mem mem_;
  std::mutex mu_;
  std::map<Key, Entry> entries_;
};

}  // namespace simp
