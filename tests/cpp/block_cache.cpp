// The kept device blocks' rules (kokkos_amd/csrc/block_cache.hpp) against a
// model of the HIP calls they use, on the host.  argv[1] names one check.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <thread>

#include "block_cache.hpp"

#define CHECK(x)                                                   \
  do {                                                             \
    if (!(x)) {                                                    \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);          \
      return 1;                                                    \
    }                                                              \
  } while (0)

constexpr size_t MiB = size_t(1) << 20;
constexpr int kUnsupported = 900;

// Addresses without memory behind them; like hipMalloc, nothing for 0 bytes.
// pending[d]: whether device d has queued work that may use any block.
struct Model {
  static constexpr int kInvalid = 1, kNoMemory = 2;
  struct Alloc {
    size_t bytes;
    int device;
  };
  static inline std::map<void*, Alloc> allocated;
  static inline uintptr_t next  = 1 << 20;
  static inline size_t capacity = size_t(64) << 30, used = 0;
  static inline int allocs = 0, frees = 0;
  static inline bool pending[2] = {};
  static inline thread_local int current = 0;
  static inline thread_local bool recording = false;  // this thread records a stream
  static int alloc(void** ptr, size_t bytes) {
    *ptr = nullptr;
    if (recording) return kUnsupported;
    if (bytes == 0) return 0;
    if (bytes > capacity - used) return kNoMemory;
    *ptr = reinterpret_cast<void*>(next);
    next += (bytes + MiB) / MiB * MiB;
    allocated[*ptr] = {bytes, current};
    used += bytes;
    ++allocs;
    return 0;
  }
  static int free(void* ptr) {
    if (recording) return kUnsupported;
    auto it = allocated.find(ptr);
    if (it == allocated.end()) return kInvalid;
    pending[it->second.device] = false;
    used -= it->second.bytes;
    allocated.erase(it);
    ++frees;
    return 0;
  }
  static int device(int* id) {
    *id = current;
    return 0;
  }
  static int set_device(int id) {
    current = id;
    return 0;
  }
  static void clear_error() {}
};
using Cache = BlockCache<Model>;

// No size wraps around to a small one, and impossible ones are refused.
int huge_requests() {
  for (size_t n : {size_t(1), size_t(4096), size_t(4097), MiB, MiB + 1, ~size_t(0) - 70000, ~size_t(0) - 65536,
                   ~size_t(0) - 65535, ~size_t(0) - 42, ~size_t(0)}) {
    CHECK(Cache::rounded(n) >= n);
    if (n < MiB * MiB) CHECK(Cache::rounded(n) - n < 65536);
  }
  Cache c;
  for (size_t n : {~size_t(0), ~size_t(0) - 42, ~size_t(0) - 65535, ~size_t(0) / 2}) {
    void* p = &c;
    CHECK(c.take(&p, n) == Model::kNoMemory);
    CHECK(p == nullptr);
  }
  return 0;
}

// A free waits for the block's device from a thread on another one, and the
// block goes to threads on its device only.
int devices() {
  Cache c;
  void *p = nullptr, *q = nullptr, *r = nullptr;
  Model::current = 1;
  CHECK(c.take(&p, MiB) == 0);
  Model::pending[0] = Model::pending[1] = true;
  int rc = -1, device = -1;
  std::thread([&] {
    rc     = c.give(p);
    device = Model::current;
  }).join();
  CHECK(rc == 0 && device == 0);
  CHECK(!Model::pending[1]);
  Model::current = 0;
  CHECK(c.take(&q, MiB) == 0);
  CHECK(q != p);
  Model::current = 1;
  CHECK(c.take(&r, MiB) == 0);
  CHECK(r == p);
  return 0;
}

// A thread that records a stream gets the answer of the call it stands for,
// and the block can be freed afterwards; a recording elsewhere changes nothing
// (the model has no call that would wait for a device by itself).
int recording() {
  Cache c;
  void* p = nullptr;
  CHECK(c.take(&p, MiB) == 0);
  Model::recording = true;
  CHECK(c.give(p) == kUnsupported);
  int rc = -1;
  std::thread([&] {
    void* q = nullptr;
    rc      = c.take(&q, 2 * MiB) || c.give(q);
  }).join();
  CHECK(rc == 0 && c.idle.size() == 1);
  Model::recording = false;
  CHECK(c.give(p) == 0);
  return 0;
}

// A block freed in stream order leaves no size behind for the block that the
// stream's allocator next makes at its address.
int freed_in_stream_order() {
  Cache c;
  void* p = nullptr;
  CHECK(c.take(&p, 64 * MiB) == 0);
  c.forget(p);
  CHECK(Model::free(p) == 0);
  Model::allocated[p] = {MiB, 0};  // the smaller one
  Model::used += MiB;
  CHECK(c.give(p) == 0);
  CHECK(c.idle.empty() && Model::allocated.count(p) == 0);
  return 0;
}

// A second free of a kept block is an error and leaves it kept, until it is
// handed out again.
int freed_twice() {
  Cache c;
  void *p = nullptr, *q = nullptr;
  CHECK(c.take(&p, MiB) == 0);
  CHECK(c.give(p) == 0);
  CHECK(c.give(p) == Model::kInvalid);
  CHECK(c.forget(p) == Model::kInvalid);
  CHECK(Model::allocated.count(p) == 1);
  CHECK(c.take(&q, MiB) == 0 && q == p);
  CHECK(c.give(q) == 0);
  c.trim();
  CHECK(c.give(q) == Model::kInvalid);
  CHECK(c.blocks.empty() && c.idle_bytes == 0 && Model::used == 0);
  return 0;
}

// Kept blocks go back where an allocation finds no memory, one of the cache's
// own or a stream-ordered one, and only there.
int no_memory() {
  Cache c;
  void *p = nullptr, *q = nullptr;
  Model::capacity = Model::used + 200 * MiB;
  CHECK(c.take(&p, 150 * MiB) == 0 && c.give(p) == 0 && c.idle.size() == 1);
  CHECK(c.take(&q, 100 * MiB) == 0);  // not of the kept block's size
  CHECK(c.idle.empty() && c.give(q) == 0 && c.idle.size() == 1);
  int calls       = 0;
  const auto pool = [&] {
    ++calls;
    return Model::alloc(&p, 150 * MiB);
  };
  CHECK(c.with_room(pool) == 0 && calls == 2 && c.idle.empty());
  q = p;
  CHECK(c.with_room(pool) == Model::kNoMemory && calls == 3);  // nothing to give back
  CHECK(Model::free(q) == 0);
  // an error of another kind, and blocks that cannot be freed now: they stay
  CHECK(c.take(&q, 100 * MiB) == 0 && c.give(q) == 0);
  Model::recording = true;
  CHECK(c.take(&p, 50 * MiB) == kUnsupported && c.with_room(pool) == kUnsupported);
  CHECK(!c.trim() && c.idle.size() == 1 && c.idle_bytes == 100 * MiB);
  Model::recording = false;
  CHECK(c.trim() && c.idle.empty() && c.idle_bytes == 0 && Model::used == 0);
  return 0;
}

// A kept block serves requests of 80-100 % of its size, at most 256 MiB are
// kept of one block and 512 MiB of all, and trim gives everything back.
int rules() {
  Cache c;
  void *p = nullptr, *q = nullptr;
  CHECK(c.take(&p, 100 * MiB) == 0 && c.give(p) == 0);
  CHECK(c.take(&q, 79 * MiB) == 0 && q != p && c.give(q) == 0);
  CHECK(c.take(&q, 101 * MiB) == 0 && q != p && c.give(q) == 0);
  c.trim();
  CHECK(c.take(&p, 100 * MiB) == 0 && c.give(p) == 0);
  CHECK(c.take(&q, 80 * MiB) == 0 && q == p && c.give(q) == 0);
  CHECK(c.take(&q, 100 * MiB) == 0 && q == p && c.give(q) == 0);
  CHECK(c.idle_bytes == 100 * MiB && c.idle.size() == 1);
  CHECK(c.take(&p, 256 * MiB) == 0 && c.take(&q, 256 * MiB + 1) == 0);
  Model::pending[0] = true;
  CHECK(c.give(q) == 0 && !Model::pending[0] && Model::allocated.count(q) == 0);
  CHECK(c.give(p) == 0 && c.idle_bytes == 356 * MiB);
  void* many[5];
  for (void*& m : many) CHECK(c.take(&m, 40 * MiB) == 0);
  for (void* m : many) CHECK(c.give(m) == 0);
  CHECK(c.idle_bytes == 476 * MiB && c.idle.size() == 5);
  CHECK(c.trim() && c.idle_bytes == 0 && Model::used == 0 && c.blocks.empty());
  CHECK(!c.trim());
  return 0;
}

int main(int argc, char** argv) {
  const struct {
    const char* name;
    int (*run)();
  } checks[] = {{"huge_requests", huge_requests}, {"devices", devices}, {"recording", recording},
                {"freed_in_stream_order", freed_in_stream_order},
                {"freed_twice", freed_twice},
                {"no_memory", no_memory}, {"rules", rules}};
  for (const auto& c : checks)
    if (argc > 1 && !std::strcmp(argv[1], c.name)) return c.run();
  std::printf("no such check\n");
  return 2;
}
