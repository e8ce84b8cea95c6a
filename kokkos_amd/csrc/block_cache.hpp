// Device blocks allocated without a stream (Views, workspaces, buffers of C
// callers).  hipMalloc and hipFree map and unmap the block's pages: a BinSort
// of 2^24 keys, which makes and releases Views of 64, 4 and 4 MiB, takes 1.97
// ms with them and 1.40 without.  A freed block is therefore kept, up to
// kIdleBytes in all and kBlockBytes each, and handed out again for a request
// of 80-100 % of its size.
//  * mx_free without a stream keeps hipFree's meaning: it returns when the
//    block's device has run everything queued before it, on any stream, so a
//    kept block is idle whoever takes it next.  That device need not be the
//    freeing thread's own: a thread starts on device 0, whichever mx_init chose.
//    The wait is that of a hipFree, of a page on the block's device (1.3 us when
//    it is idle): hipDeviceSynchronize would invalidate a stream capture that
//    another thread is in, which freeing memory there does not.
//  * A block is handed out only to threads on its device.
//  * Kept blocks go back to the device when an allocation, also a stream-ordered
//    one, finds no memory, by mx_trim (Kokkos::finalize calls it) and at
//    mx_finalize.
//  * A thread that is recording a stream gets what hipFree answers there.
//
// Api stands for the HIP calls, as static functions that return 0 or an error:
//   alloc(ptr*, bytes), free(ptr), device(id*), set_device(id), clear_error()
// and the errors kInvalid of an argument that cannot be and kNoMemory.
// alloc and set_device are about the calling thread's device; free waits for the
// device of ptr.
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
  struct Block {
    int device;
    size_t bytes;
    bool operator<(const Block& o) const { return device != o.device ? device < o.device : bytes < o.bytes; }
  };
  struct State : Block {
    bool freed;  // by the caller: kept, or on the way there
  };
  std::unordered_map<void*, State> blocks;  // the callers' and the kept ones
  std::multimap<Block, void*> idle;
  size_t idle_bytes = 0;

  // Sizes that would wrap stay as they are, for the allocation to refuse.
  static size_t rounded(size_t n) {
    const size_t unit = n <= (size_t(1) << 20) ? size_t(4) << 10 : size_t(64) << 10;
    return n > ~size_t(0) - unit ? n : (n + unit - 1) / unit * unit;
  }
  // With mtx held.  Returns whether any block went back; one that cannot be
  // freed now (this thread is recording) stays.
  bool release_idle() {
    bool any = false;
    for (auto it = idle.begin(); it != idle.end();) {
      if (Api::free(it->second) != 0) {
        Api::clear_error();
        ++it;
        continue;
      }
      any = true;
      idle_bytes -= it->first.bytes;
      blocks.erase(it->second);
      it = idle.erase(it);
    }
    return any;
  }
  bool trim() {
    std::lock_guard<std::mutex> lk(mtx);
    return release_idle();
  }
  int take(void** ptr, size_t bytes) {
    *ptr              = nullptr;
    const size_t want = rounded(bytes);
    int device        = 0;
    if (const int e = Api::device(&device)) return e;
    std::lock_guard<std::mutex> lk(mtx);
    auto it = idle.lower_bound({device, want});
    if (it != idle.end() && it->first.device == device && it->first.bytes <= want + want / 4) {
      *ptr         = it->second;
      blocks[*ptr] = {it->first, false};
      idle_bytes -= it->first.bytes;
      idle.erase(it);
      return 0;
    }
    int e = Api::alloc(ptr, want);
    if (e == Api::kNoMemory && !idle.empty()) {
      Api::clear_error();
      if (release_idle()) e = Api::alloc(ptr, want);
    }
    if (e == 0) blocks[*ptr] = {{device, want}, false};
    else *ptr = nullptr;
    return e;
  }
  // An allocation that is not for the cache: `alloc` again after the kept blocks
  // went back, where it found no memory.
  template <class F>
  int with_room(const F& alloc) {
    const int e = alloc();
    if (e != Api::kNoMemory || !trim()) return e;
    Api::clear_error();
    return alloc();
  }
  // The block leaves by another way (a stream-ordered free): its size must not
  // stay for another block at its address.
  int forget(void* ptr) {
    std::lock_guard<std::mutex> lk(mtx);
    auto it = blocks.find(ptr);
    if (it == blocks.end()) return 0;
    if (it->second.freed) return Api::kInvalid;
    blocks.erase(it);
    return 0;
  }
  // Waits for `device`, from a thread on any device.
  static int wait_for(int device) {
    int mine = 0;
    if (const int e = Api::device(&mine)) return e;
    if (mine != device)
      if (const int e = Api::set_device(device)) return e;
    void* page  = nullptr;
    const int e = Api::alloc(&page, 4096);
    if (mine != device) (void)Api::set_device(mine);
    return e ? e : Api::free(page);
  }
  // A block that is freed a second time is refused, as hipFree does.
  int give(void* ptr) {
    State b{{0, 0}, false};
    {
      std::lock_guard<std::mutex> lk(mtx);
      auto it = blocks.find(ptr);
      if (it != blocks.end()) {
        if (it->second.freed) return Api::kInvalid;
        it->second.freed = true;
        b                = it->second;
      }
    }
    if (b.bytes == 0) return Api::free(ptr);
    const bool keep   = b.bytes <= kBlockBytes;
    const bool waited = keep && wait_for(b.device) == 0;
    if (keep && !waited) Api::clear_error();
    {
      std::lock_guard<std::mutex> lk(mtx);
      if (waited && idle_bytes + b.bytes <= kIdleBytes) {
        idle.emplace(b, ptr);
        idle_bytes += b.bytes;
        return 0;
      }
      blocks.erase(ptr);
    }
    return Api::free(ptr);
  }
};

#endif
