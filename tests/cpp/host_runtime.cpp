// A stand-in for libkkmx_rt.so without a GPU: memory is the host's, launches
// are recorded and not run.  With it the host side of the dispatches in
// libkkmx_paths.so runs on the CPU (tests/host_runtime.py).  It is also a
// Kokkos tool that notes the labels of parallel_for, and on request a tuning
// tool that answers nothing.
#include <dlfcn.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "kkmx_runtime.h"

namespace {
struct Launch {
  std::string kernel;
  uint64_t grid, block;
  std::string args;  // the first byte of each
};
std::vector<Launch> launches;
std::vector<std::string> labels;
std::map<void*, size_t> blocks;
size_t limit   = ~size_t(0);  // of one allocation
int cus        = 256;
int capturing  = 0;
int allocs     = 0;
int one_stream = 0, one_event = 0;
int take(void** p, size_t n) {
  *p = nullptr;
  if (n == 0) return 0;
  if (n > limit) return 2;
  *p = std::calloc(n, 1);
  if (!*p) return 2;
  blocks[*p] = n;
  ++allocs;
  return 0;
}
int give(void* p) {
  if (p && blocks.erase(p) == 0) return 1;
  std::free(p);
  return 0;
}
}  // namespace

extern "C" {
// ---- what a test sets and reads
void host_set_cus(int n) { cus = n; }
void host_set_limit(size_t n) { limit = n; }
void host_set_capturing(int yes) { capturing = yes; }
void host_clear() {
  launches.clear();
  labels.clear();
  allocs = 0;
}
int host_launches() { return int(launches.size()); }
const char* host_kernel(int i) { return launches[i].kernel.c_str(); }
uint64_t host_grid(int i) { return launches[i].grid; }
uint64_t host_block(int i) { return launches[i].block; }
int host_args(int i) { return int(launches[i].args.size()); }
int host_arg(int i, int arg) { return static_cast<unsigned char>(launches[i].args[arg]); }
int host_labels() { return int(labels.size()); }
const char* host_label(int i) { return labels[i].c_str(); }
int host_allocs() { return allocs; }
size_t host_held() {
  size_t n = 0;
  for (auto& b : blocks) n += b.second;
  return n;
}

// ---- Kokkos Tools
void kokkosp_begin_parallel_for(const char* name, uint32_t, uint64_t* id) {
  *id = 0;
  labels.push_back(name);
}
void kokkosp_end_parallel_for(uint64_t) {}

// ---- the runtime
int mx_init(int) { return 0; }
int mx_finalize(void) { return 0; }
int mx_is_initialized(void) { return 1; }
int mx_device_count(int* n) {
  *n = 1;
  return 0;
}
int mx_device_props_get(mx_device_props* p) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->name, "host");
  std::strcpy(p->arch, "gfx950");
  p->cu_count              = cus;
  p->wave_size             = 64;
  p->max_threads_per_block = 1024;
  p->max_threads_per_cu    = 2048;
  p->regs_per_block        = 65536;
  p->xcc_count             = 8;
  p->lds_per_block = p->lds_per_cu = 160 * 1024;
  p->global_mem                    = size_t(288) << 30;
  p->max_grid_x                    = 0x7fffffff;
  return 0;
}
int mx_current_device(int* d) {
  *d = 0;
  return 0;
}
int mx_malloc(void** p, size_t n, mx_stream_t) { return take(p, n); }
int mx_free(void* p, mx_stream_t) { return give(p); }
int mx_trim(void) { return 0; }
int mx_host_alloc(void** p, size_t n) { return take(p, n); }
int mx_host_free(void* p) { return give(p); }
int mx_pointer_kind(const void*, int* kind) {
  *kind = 1;
  return 0;
}
int mx_memcpy_async(void* d, const void* s, size_t n, mx_stream_t) {
  std::memmove(d, s, n);
  return 0;
}
int mx_memcpy(void* d, const void* s, size_t n) {
  std::memmove(d, s, n);
  return 0;
}
int mx_memset_async(void* d, int v, size_t n, mx_stream_t) {
  std::memset(d, v, n);
  return 0;
}
int mx_stream_create(mx_stream_t* s) {
  *s = &one_stream;
  return 0;
}
int mx_stream_destroy(mx_stream_t) { return 0; }
int mx_stream_sync(mx_stream_t) { return capturing ? 900 : 0; }
int mx_stream_query(mx_stream_t) { return 0; }
int mx_device_sync(void) { return capturing ? 900 : 0; }
int mx_event_create(mx_event_t* e) {
  *e = &one_event;
  return 0;
}
int mx_event_destroy(mx_event_t) { return 0; }
int mx_event_record(mx_event_t, mx_stream_t) { return 0; }
int mx_event_sync(mx_event_t) { return 0; }
int mx_event_query(mx_event_t) { return 0; }
int mx_event_elapsed_ms(float* ms, mx_event_t, mx_event_t) {
  *ms = 0;
  return 0;
}
int mx_stream_capturing(mx_stream_t, int* yes) {
  *yes = capturing;
  return 0;
}
int mx_stream_wait_event(mx_stream_t, mx_event_t) { return 0; }
int mx_launch(const void* fn, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz, size_t,
              void** args, mx_stream_t) {
  std::string bytes;
  while (args && *args) bytes += *static_cast<char*>(*args++);
  Dl_info info;
  const bool known = dladdr(fn, &info) != 0 && info.dli_sname;
  launches.push_back({known ? info.dli_sname : "", uint64_t(gx) * gy * gz, uint64_t(bx) * by * bz, bytes});
  return 0;
}
int mx_func_attributes(const void*, int* threads, int* regs, size_t* lds, size_t* priv) {
  if (threads) *threads = 1024;
  if (regs) *regs = 64;
  if (lds) *lds = 0;
  if (priv) *priv = 0;
  return 0;
}
int mx_occupancy(const void*, int, size_t, int* blocks_per_cu) {
  *blocks_per_cu = 2;
  return 0;
}
int mx_get_last_error(void) { return 0; }
int mx_graph_capture_begin(mx_stream_t) { return 0; }
int mx_graph_capture_end(mx_stream_t, mx_graph_t* g) {
  *g = &one_event;
  return 0;
}
int mx_graph_instantiate(mx_graph_exec_t* e, mx_graph_t) {
  *e = &one_event;
  return 0;
}
int mx_graph_launch(mx_graph_exec_t, mx_stream_t) { return 0; }
int mx_graph_exec_destroy(mx_graph_exec_t) { return 0; }
int mx_graph_destroy(mx_graph_t) { return 0; }
int mx_graph_node_count(mx_graph_t, size_t* n) {
  *n = 0;
  return 0;
}
const char* mx_error_string(int) { return "host stand-in"; }
int mx_default_stream(mx_stream_t* s) {
  *s = &one_stream;
  return 0;
}
}
