// bins[idx[i]] += vals[i] for many FP64 values, without a device-scope atomic
// per value.
//
// A device-scope FP64 atomic on a random address leaves the XCD's L2 and runs
// at the memory side, 2.4e10 of them a second, whatever the arrangement.  Here
// the (index, value) pairs of a piece are first moved, by one pass of the
// radix sort's kernels over the top bits of the index, into up to 256 runs
// whose bins fit in LDS; then one block per run adds its values into LDS bins
// and adds those to the caller's bins, one atomic per bin and block.  Up to
// kScatterDirect bins skip the move.  2^26 values into 2^20 bins take 0.76 ms
// (2.83 by atomics): in four pieces, each 127 us of move (count 16, offsets 5,
// scatter 106) and 64 of sums; into 1000 bins 0.14 (9.4).
//
// Bins start from -0.0 in LDS, the value that changes nothing when added, and
// bins still at -0.0 are left alone, so untouched bins keep their bits.  As
// with plain atomics the order of additions to one bin is not fixed.
#ifndef KKMX_BINNEDSCATTER_HPP
#define KKMX_BINNEDSCATTER_HPP

#include <kkmx/RadixSort.hpp>

namespace Kokkos {
namespace Impl {

constexpr int kScatterLanes       = 1024;
constexpr int kScatterMaxShift    = 13;       // log2 of the bins of a run: 64 KiB of LDS, two blocks per CU
constexpr int kScatterDirect      = 1 << 12;  // bins
constexpr int64_t kScatterMaxBins = int64_t(256) << kScatterMaxShift;
// Values per piece: 192 MiB of workspace, which the memory-side cache holds.
constexpr int64_t kScatterPiece = int64_t(1) << 24;
// The move and its four launches pay from about 2^20 values: 2^20 into 2^20
// bins take 49 us by atomics and 32 binned, 2^19 into 10^5 bins 27 and 25.
// Few bins pay from 2^18: atomics on them wait for one another (2^19 into 1000
// bins 78 us and 17).
constexpr int64_t kScatterMin       = int64_t(1) << 20;
constexpr int64_t kScatterDirectMin = int64_t(1) << 18;

// One part of one run: `part` values of it at most.  totals[d] is the number
// of values of run d; without them (direct) everything is run 0.  HBM bounds
// it, 12 bytes a value, with 8 pairs of loads in flight per lane.
template <class Unused = void>
__global__ __launch_bounds__(kScatterLanes) void k_scatter_bins(const uint32_t* idx, const double* vals, const int64_t n,
                                                                const uint32_t* totals, const int64_t part,
                                                                const int bin_shift, double* bins, const int64_t nbins) {
  extern __shared__ __align__(16) unsigned char kkmx_dyn_lds[];
  double* acc = reinterpret_cast<double*>(kkmx_dyn_lds);
  __shared__ uint32_t s_wave[4], s_run, s_first, s_count;
  const int t = threadIdx.x;
  if (t == 0) s_count = 0;
  __syncthreads();
  if (totals) {
    const uint32_t mine  = t < 256 ? totals[t] : 0u;
    const uint32_t parts = uint32_t((int64_t(mine) + part - 1) / part);
    const uint32_t first = radix_prefix256<16>(mine, s_wave);
    __syncthreads();
    const uint32_t before = radix_prefix256<16>(parts, s_wave);
    if (t < 256 && blockIdx.x >= before && blockIdx.x < before + parts) {
      const int64_t skip = int64_t(blockIdx.x - before) * part;
      s_run              = uint32_t(t);
      s_first            = first + uint32_t(skip);
      s_count            = uint32_t(mine - skip < part ? mine - skip : part);
    }
  } else if (t == 0) {
    const int64_t skip = int64_t(blockIdx.x) * part;
    s_run              = 0;
    s_first            = uint32_t(skip);
    s_count            = uint32_t(n - skip < part ? n - skip : part);
  }
  __syncthreads();
  const uint32_t count = s_count;
  if (count == 0) return;
  const int width = totals ? 1 << bin_shift : int(nbins);
  for (int b = t; b < width; b += kScatterLanes) acc[b] = -0.0;
  __syncthreads();
  const uint32_t mask = totals ? uint32_t(width - 1) : ~0u;
  const uint32_t* at  = idx + s_first;
  const double* from  = vals + s_first;
  constexpr int Items = 8;
  for (uint32_t b = 0; b < count; b += kScatterLanes * Items) {
    uint32_t k[Items];
    double x[Items];
#pragma unroll
    for (int r = 0; r < Items; ++r) {
      const uint32_t i = b + r * kScatterLanes + t;
      k[r]             = i < count ? at[i] & mask : ~0u;
      x[r]             = i < count ? from[i] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < Items; ++r)
      if (k[r] < uint32_t(width)) __hip_atomic_fetch_add(&acc[k[r]], x[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __syncthreads();
  const int64_t bin0 = int64_t(s_run) << bin_shift;
  for (int b = t; b < width; b += kScatterLanes) {
    const double v = acc[b];
    if (__double_as_longlong(v) != __double_as_longlong(-0.0) && bin0 + b < nbins) atomic_add(&bins[bin0 + b], v);
  }
}

// The moved pairs of a piece and the counts, kept between calls, at most
// kScatterPiece pairs; freed by Kokkos::finalize.  Every use is ordered on the
// default instance's stream, and the mutex keeps one call's launches together.
struct ScatterWorkspace {
  std::mutex mtx;
  void* buf     = nullptr;
  size_t bytes  = 0;
  bool hooked   = false;
};
inline ScatterWorkspace& scatter_workspace() {
  static ScatterWorkspace w;
  return w;
}
inline void scatter_workspace_release() {
  ScatterWorkspace& w = scatter_workspace();
  std::lock_guard<std::mutex> lock(w.mtx);
  if (w.buf) KKMX_SAFE_CALL(mx_free(w.buf, nullptr));
  w.buf    = nullptr;
  w.bytes  = 0;
  w.hooked = false;
}

// Whether binned_scatter_add takes a call: not while the stream is captured (a
// graph would keep the workspace's address), nor where the atomics are faster.
inline bool binned_scatter_takes(int64_t n, int64_t nbins, mx_stream_t stream) {
  if (n < (nbins <= kScatterDirect ? kScatterDirectMin : kScatterMin) || nbins > kScatterMaxBins) return false;
  int capturing = 0;
  return mx_stream_capturing(stream, &capturing) == 0 && !capturing;
}

// bins[idx[i]] += vals[i], i < n, on the default instance; to a tool, one
// parallel_for by the name of `label`, as the atomics are.  False, with nothing
// done, where there is no memory for the workspace: atomics need none.
inline bool binned_scatter_add(const char* label, const double* vals, const int32_t* idx, int64_t n, double* bins,
                               int64_t nbins) {
  MI355X exec;
  mx_stream_t stream = exec.stream();
  const int cus      = MI355X::impl_cu_count() > 0 ? MI355X::impl_cu_count() : 256;
  const uint32_t* k0 = reinterpret_cast<const uint32_t*>(idx);
  const void* kernel = reinterpret_cast<const void*>(&k_scatter_bins<>);
  if (nbins <= kScatterDirect) {
    const ToolsKernel<MI355X> tools(label, exec, 0);
    // two blocks per CU, and a round of the lanes each; pieces keep the
    // positions 32-bit
    for (int64_t done = 0; done < n;) {
      int64_t m              = n - done < (int64_t(1) << 30) ? n - done : int64_t(1) << 30;
      int64_t part           = (m + 2 * cus - 1) / (2 * cus);
      if (part < 8192) part = 8192;
      const uint32_t* i0     = k0 + done;
      const double* v0       = vals + done;
      const uint32_t* totals = nullptr;
      int bin_shift          = 0;
      mx_launch_kernel(kernel, unsigned((m + part - 1) / part), kScatterLanes, size_t(nbins) * sizeof(double), stream,
                       i0, v0, m, totals, part, bin_shift, bins, nbins);
      done += m;
    }
    return true;
  }
  int bin_shift = 10;  // at least 1024 bins a run: fewer would meet in LDS
  while ((nbins - 1) >> bin_shift > 255) ++bin_shift;
  using Shape              = RadixShape<uint32_t, uint64_t, true>;
  constexpr int tile       = Shape::lanes * Shape::items;
  const int64_t pieces     = (n + kScatterPiece - 1) / kScatterPiece;
  const int64_t piece      = (n + pieces - 1) / pieces;
  const size_t key_bytes   = radix_round(size_t(piece) * sizeof(uint32_t));
  const size_t val_bytes   = radix_round(size_t(piece) * sizeof(double));
  const size_t count_bytes = size_t(cus) * Shape::blocks * 256 * sizeof(uint32_t);
  const size_t need        = key_bytes + val_bytes + count_bytes + sizeof(RadixControl);
  ScatterWorkspace& ws     = scatter_workspace();
  std::lock_guard<std::mutex> lock(ws.mtx);
  if (ws.bytes < need) {
    if (ws.buf) KKMX_SAFE_CALL(mx_free(ws.buf, nullptr));
    ws.buf   = nullptr;
    ws.bytes = 0;
    if (mx_malloc(&ws.buf, need, nullptr) != 0) {
      (void)mx_get_last_error();
      return false;
    }
    ws.bytes = need;
  }
  if (!ws.hooked) {
    push_finalize_hook(&scatter_workspace_release);
    ws.hooked = true;
  }
  const ToolsKernel<MI355X> tools(label, exec, 0);
  char* base        = static_cast<char*>(ws.buf);
  uint32_t* k1      = reinterpret_cast<uint32_t*>(base);
  uint64_t* v1      = reinterpret_cast<uint64_t*>(base + key_bytes);
  uint32_t* counts  = reinterpret_cast<uint32_t*>(base + key_bytes + val_bytes);
  RadixControl* ctl = reinterpret_cast<RadixControl*>(base + key_bytes + val_bytes + count_bytes);
  int pass = -1, turn = 0;
  bool fold = false, summed = true;  // k_scatter_bins reads the totals, so k_radix_offsets always runs
  for (int64_t done = 0; done < n; done += piece) {
    int64_t m              = n - done < piece ? n - done : piece;
    const uint32_t* i0     = k0 + done;
    const uint64_t* v0     = reinterpret_cast<const uint64_t*>(vals + done);
    const int64_t ntiles   = (m + tile - 1) / tile;
    const int64_t tpb      = (ntiles + int64_t(cus) * Shape::blocks - 1) / (int64_t(cus) * Shape::blocks);
    int64_t segment        = tpb * tile;
    int segments           = int((ntiles + tpb - 1) / tpb);
    mx_launch_kernel(reinterpret_cast<const void*>(&k_radix_count<uint32_t, false>), unsigned(segments),
                     kRadixCountLanes, 0, stream, pass, bin_shift, m, segment, i0, k1, ctl, turn, fold, counts);
    mx_launch_kernel(reinterpret_cast<const void*>(&k_radix_offsets<uint32_t, false>), 64, kRadixOffsetLanes, 0, stream,
                     pass, ctl, turn, counts, segments);
    mx_launch_kernel(
        reinterpret_cast<const void*>(&k_radix_scatter<uint32_t, uint64_t, false, Shape::lanes, Shape::items>),
        unsigned(segments), Shape::lanes, 0, stream, pass, bin_shift, m, segment, i0, k1, v0, v1, ctl, turn, counts,
        summed);
    // a part of an evenly filled run is the whole run
    int64_t part           = m / 256 + m / 2048 + 1;
    const uint32_t* totals = ctl->totals;
    const uint32_t* ck1    = k1;
    const double* cv1      = reinterpret_cast<const double*>(v1);
    mx_launch_kernel(kernel, unsigned(256 + (m + part - 1) / part), kScatterLanes, sizeof(double) << bin_shift, stream,
                     ck1, cv1, m, totals, part, bin_shift, bins, nbins);
  }
  return true;
}

}  // namespace Impl
}  // namespace Kokkos

#endif
