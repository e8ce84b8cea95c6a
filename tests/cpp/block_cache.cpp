// The kept device blocks' rules (kokkos_amd/csrc/block_cache.hpp) against a
// model of the HIP calls they use, on the host.  argv[1] names one check.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>

#include "block_cache.hpp"

#define CHECK(x)                                                   \
  do {                                                             \
    if (!(x)) {                                                    \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);          \
      return 1;                                                    \
    }                                                              \
  } while (0)

constexpr size_t MiB = size_t(1) << 20;
constexpr int kInvalid = 1, kNoMemory = 2;

// Addresses without memory behind them; like hipMalloc, nothing for 0 bytes.
struct Model {
  static inline std::map<void*, size_t> allocated;
  static inline uintptr_t next    = 1 << 20;
  static inline size_t capacity   = size_t(64) << 30, used = 0;
  static inline int allocs = 0, frees = 0;
  static int alloc(void** ptr, size_t bytes) {
    *ptr = nullptr;
    if (bytes == 0) return 0;
    if (bytes > capacity - used) return kNoMemory;
    *ptr = reinterpret_cast<void*>(next);
    next += (bytes + MiB) / MiB * MiB;
    allocated[*ptr] = bytes;
    used += bytes;
    ++allocs;
    return 0;
  }
  static int free(void* ptr) {
    auto it = allocated.find(ptr);
    if (it == allocated.end()) return kInvalid;
    used -= it->second;
    allocated.erase(it);
    ++frees;
    return 0;
  }
  static int sync() { return 0; }
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
    CHECK(c.take(&p, n) == kNoMemory);
    CHECK(p == nullptr);
  }
  return 0;
}

int main(int argc, char** argv) {
  const struct {
    const char* name;
    int (*run)();
  } checks[] = {{"huge_requests", huge_requests}};
  for (const auto& c : checks)
    if (argc > 1 && !std::strcmp(argv[1], c.name)) return c.run();
  std::printf("no such check\n");
  return 2;
}
