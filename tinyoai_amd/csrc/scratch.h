// Which device buffer a product's operand planes and partials take: never one
// that work on another stream, or of another graph, may still use. Plain host
// code; the caller brings the allocation.
#pragma once

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <functional>
#include <map>
#include <utility>
#include <vector>

namespace tinyoai {

class ScratchPool {
 public:
  using Alloc = std::function<void *(size_t)>;  // null: out of memory
  using Free = std::function<void(void *)>;
  // Streams with a buffer of their own; those past them share one buffer,
  // whose users the caller orders one after another.
  static constexpr size_t kStreams = 8;

  struct Lease {
    void *ptr = nullptr;
    bool shared = false;
  };
  // A captured buffer: in use until its graph, and every executable graph made
  // from it, has let go of the record (release, which may run on any thread,
  // before or after the pool's end).
  struct Record {
    void *ptr = nullptr;
    size_t bytes = 0;
    std::atomic<int> owners{2};  // the pool and the graph
    std::atomic<bool> used{true};
  };
  static void release(void *record) {
    Record *r = static_cast<Record *>(record);
    r->used.store(false, std::memory_order_release);
    drop(r);
  }

  // For work enqueued on `stream` (and, where one handle names a stream of
  // each thread, on thread `thread`'s), which runs in order there. A buffer
  // that has become too small is kept: enqueued work may still use it (each
  // is at least half as large again, so all of them are no more than three
  // times the last).
  Lease eager(const void *stream, uint64_t thread, size_t bytes, const Alloc &alloc) {
    auto it = streams_.find({stream, thread});
    const bool shared = it == streams_.end() && streams_.size() >= kStreams;
    if (it == streams_.end() && !shared) it = streams_.emplace(Key{stream, thread}, Buffer{}).first;
    Buffer &b = shared ? shared_ : it->second;
    if (b.bytes < bytes) {
      size_t want = bytes > b.bytes + b.bytes / 2 ? bytes : b.bytes + b.bytes / 2;
      kept_.reserve(kept_.size() + 1);
      void *p = alloc(want);
      if (!p && want > bytes) p = alloc(want = bytes);
      if (!p) return Lease{};
      if (b.ptr) kept_.push_back(b.ptr);
      b = Buffer{p, want};
    }
    return Lease{b.ptr, shared};
  }

  // For work captured on `stream` by the capture `id`: the buffer that this
  // capture took there before, where it is large enough; else one that a
  // destroyed graph has let go of, or a new one, and then *made is its record,
  // to be given to the graph (or released, if that fails).
  void *captured(uint64_t id, const void *stream, size_t bytes, const Alloc &alloc, Record **made) {
    *made = nullptr;
    for (auto &c : captures_)
      if (c.id == id && c.stream == stream && c.record->bytes >= bytes && c.record->used.load(std::memory_order_acquire))
        return c.record->ptr;
    captures_.reserve(captures_.size() + 1);
    for (auto &c : captures_)
      if (c.record->bytes >= bytes && !c.record->used.load(std::memory_order_acquire)) {
        Record *r = new Record;
        r->ptr = c.record->ptr;
        r->bytes = c.record->bytes;
        drop(c.record);
        c = Capture{id, stream, r};
        *made = r;
        return r->ptr;
      }
    Record *r = new Record;
    r->ptr = alloc(bytes);
    r->bytes = bytes;
    if (!r->ptr) {
      delete r;
      return nullptr;
    }
    captures_.push_back(Capture{id, stream, r});
    *made = r;
    return r->ptr;
  }

  // Every buffer given back; no work may use them any more.
  void clear(const Free &free) {
    for (auto &s : streams_)
      if (s.second.ptr) free(s.second.ptr);
    if (shared_.ptr) free(shared_.ptr);
    for (void *p : kept_) free(p);
    for (auto &c : captures_) {
      free(c.record->ptr);
      drop(c.record);
    }
    streams_.clear();
    shared_ = Buffer{};
    kept_.clear();
    captures_.clear();
  }

 private:
  using Key = std::pair<const void *, uint64_t>;
  struct Buffer {
    void *ptr = nullptr;
    size_t bytes = 0;
  };
  struct Capture {
    uint64_t id;
    const void *stream;
    Record *record;
  };
  static void drop(Record *r) {
    if (r->owners.fetch_sub(1, std::memory_order_acq_rel) == 1) delete r;
  }
  std::map<Key, Buffer> streams_;
  Buffer shared_;
  std::vector<void *> kept_;
  std::vector<Capture> captures_;
};

}  // namespace tinyoai
