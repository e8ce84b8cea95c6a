// Device blocks allocated without a stream (Views, workspaces, buffers of C
// callers).  hipMalloc and hipFree map and unmap the block's pages: a BinSort
// of 2^24 keys, which makes and releases Views of 64, 4 and 4 MiB, takes 1.97
// ms with them and 1.40 without.  A freed block is therefore kept, up to
// kIdleBytes in all and kBlockBytes each, and handed out again for a request
// of 80-100 % of its size.
//  * mx_free without a stream keeps hipFree's meaning: it returns when the
//    device has run everything queued before it, on any stream, so a kept
//    block is idle whoever takes it next.
//  * Kept blocks go back to the device when an allocation fails, by mx_trim
//    (Kokkos::finalize calls it) and at mx_finalize.
//  * A thread that is recording a stream goes to hipFree as before: waiting
//    for the device is not allowed there.
//
// Api stands for the HIP calls, as static functions that return 0 or an error:
//   alloc(ptr*, bytes), free(ptr), sync(), clear_error()
#ifndef KKMX_BLOCK_CACHE_HPP
#define KKMX_BLOCK_CACHE_HPP

#include <cstddef>
#include <map>
#include <mutex>
#include <unordered_map>

template <class Api>
struct BlockCache {
  static constexpr size_t kBlockBytes = size_t(256) << 20;
  static constexpr size_t kIdleBytes  = size_t(512) << 20;
  std::mutex mtx;
  std::unordered_map<void*, size_t> live;
  std::multimap<size_t, void*> idle;
  size_t idle_bytes = 0;

  // Sizes that would wrap stay as they are, for the allocation to refuse.
  static size_t rounded(size_t n) {
    const size_t unit = n <= (size_t(1) << 20) ? size_t(4) << 10 : size_t(64) << 10;
    return n > ~size_t(0) - unit ? n : (n + unit - 1) / unit * unit;
  }
  // with mtx held
  void release_idle() {
    for (auto& b : idle) (void)Api::free(b.second);
    idle.clear();
    idle_bytes = 0;
  }
  void trim() {
    std::lock_guard<std::mutex> lk(mtx);
    release_idle();
  }
  int take(void** ptr, size_t bytes) {
    const size_t want = rounded(bytes);
    std::lock_guard<std::mutex> lk(mtx);
    auto it = idle.lower_bound(want);
    if (it != idle.end() && it->first <= want + want / 4) {
      *ptr       = it->second;
      live[*ptr] = it->first;
      idle_bytes -= it->first;
      idle.erase(it);
      return 0;
    }
    int e = Api::alloc(ptr, want);
    if (e != 0 && !idle.empty()) {
      Api::clear_error();
      release_idle();
      e = Api::alloc(ptr, want);
    }
    if (e == 0) live[*ptr] = want;
    else *ptr = nullptr;
    return e;
  }
  int give(void* ptr, bool recording) {
    size_t bytes = 0;
    {
      std::lock_guard<std::mutex> lk(mtx);
      auto it = live.find(ptr);
      if (it != live.end()) {
        bytes = it->second;
        live.erase(it);
      }
    }
    if (bytes == 0 || bytes > kBlockBytes || recording) return Api::free(ptr);
    if (Api::sync() != 0) {
      Api::clear_error();
      return Api::free(ptr);
    }
    std::lock_guard<std::mutex> lk(mtx);
    if (idle_bytes + bytes > kIdleBytes) return Api::free(ptr);
    idle.emplace(bytes, ptr);
    idle_bytes += bytes;
    return 0;
  }
};

#endif
