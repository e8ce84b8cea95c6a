// Sorting for the MI355X execution space: Kokkos::BinSort with BinOp1D /
// BinOp3D, and Kokkos::sort.
//
// Reference: algorithms/src/sorting/Kokkos_BinSortPublicAPI.hpp (BinSort:
// count keys per bin, exclusive scan of the counts into bin offsets, place
// every index at its bin's next slot, optionally sort within bins, then
// permute values through the permutation vector),
// algorithms/src/sorting/Kokkos_BinOpsPublicAPI.hpp (BinOp1D / BinOp3D:
// bin(keys, i), max_bins(), and the in-bin comparison), and
// algorithms/src/sorting/Kokkos_SortPublicAPI.hpp (sort(view),
// sort(exec, view), sort(view, comparator), sort(view, begin, end)).
//
// Kokkos::sort of a contiguous rank-1 device View of 4- or 8-byte
// arithmetic keys is the LSD radix sort of RadixSort.hpp.  As in the
// reference's HIP path (thrust::sort, a radix sort for arithmetic keys:
// algorithms/src/sorting/impl/Kokkos_SortImpl.hpp:222-240), -0.0 and +0.0
// compare equal and keep their input order, and NaNs go below -inf (sign bit
// set) or above +inf.  Other element types, comparators and host Views sort
// on the host with std::sort (results identical to an ascending sort).
#ifndef KKMX_SORT_HPP
#define KKMX_SORT_HPP

#include <Kokkos_Core.hpp>
#include <kkmx/RadixSort.hpp>

#include <algorithm>
#include <vector>

namespace Kokkos {

// ------------------------------------------------------------------ bin ops
template <class KeyViewType>
struct BinOp1D {
  int max_bins_ = 0;
  double mul_   = 0;
  double min_   = 0;
  BinOp1D() = delete;
  // max_bins bins over [min, max] (one extra bin holds max itself); integer
  // keys whose range is at most max_bins get one value per bin.
  BinOp1D(int max_bins, typename KeyViewType::const_value_type min, typename KeyViewType::const_value_type max)
      : max_bins_(max_bins + 1),
        mul_(static_cast<double>(max_bins) / (static_cast<double>(max) - static_cast<double>(min))),
        min_(static_cast<double>(min)) {
    if (std::is_integral<typename KeyViewType::non_const_value_type>::value &&
        static_cast<double>(max) - static_cast<double>(min) <= static_cast<double>(max_bins))
      mul_ = 1.0;
  }
  template <class ViewType>
  KOKKOS_INLINE_FUNCTION int bin(ViewType& keys, const int& i) const {
    return static_cast<int>(mul_ * (static_cast<double>(keys(i)) - min_));
  }
  KOKKOS_INLINE_FUNCTION int max_bins() const { return max_bins_; }
  // true: key i1 goes before key i2 inside a bin
  template <class ViewType, class I1, class I2>
  KOKKOS_INLINE_FUNCTION bool operator()(ViewType& keys, I1& i1, I2& i2) const {
    return keys(i1) < keys(i2);
  }
};

template <class KeyViewType>
struct BinOp3D {
  int max_bins_[3] = {0, 0, 0};
  double mul_[3]   = {0, 0, 0};
  double min_[3]   = {0, 0, 0};
  BinOp3D() = delete;
  BinOp3D(int max_bins[], typename KeyViewType::const_value_type min[],
          typename KeyViewType::const_value_type max[]) {
    for (int d = 0; d < 3; ++d) {
      max_bins_[d] = max_bins[d];
      mul_[d]      = static_cast<double>(max_bins[d]) / (static_cast<double>(max[d]) - static_cast<double>(min[d]));
      min_[d]      = static_cast<double>(min[d]);
    }
  }
  template <class ViewType>
  KOKKOS_INLINE_FUNCTION int bin(ViewType& keys, const int& i) const {
    const int b0 = int(mul_[0] * (keys(i, 0) - min_[0]));
    const int b1 = int(mul_[1] * (keys(i, 1) - min_[1]));
    const int b2 = int(mul_[2] * (keys(i, 2) - min_[2]));
    return (b0 * max_bins_[1] + b1) * max_bins_[2] + b2;
  }
  KOKKOS_INLINE_FUNCTION int max_bins() const { return max_bins_[0] * max_bins_[1] * max_bins_[2]; }
  // lexicographically greater first (the reference's in-bin order)
  template <class ViewType, class I1, class I2>
  KOKKOS_INLINE_FUNCTION bool operator()(ViewType& keys, I1& i1, I2& i2) const {
    for (int d = 0; d < 3; ++d) {
      if (keys(i1, d) > keys(i2, d)) return true;
      if (keys(i1, d) != keys(i2, d)) return false;
    }
    return false;
  }
};

namespace Impl {

template <class Keys, class Op>
struct BinCountF {
  Keys keys;
  Op op;
  View<int*, MI355XSpace, MemoryTraits<Unmanaged>> count;
  int begin;
  KOKKOS_INLINE_FUNCTION void operator()(const int i) const { atomic_add(&count(op.bin(keys, begin + i)), 1); }
};
struct BinOffsetF {
  View<const int*, MI355XSpace, MemoryTraits<Unmanaged>> count;
  View<int*, MI355XSpace, MemoryTraits<Unmanaged>> offsets;
  KOKKOS_INLINE_FUNCTION void operator()(const int i, int& upd, const bool final) const {
    if (final) offsets(i) = upd;
    upd += count(i);
  }
};
template <class Keys, class Op>
struct BinPlaceF {
  Keys keys;
  Op op;
  View<int*, MI355XSpace, MemoryTraits<Unmanaged>> fill;
  View<const int*, MI355XSpace, MemoryTraits<Unmanaged>> offsets;
  View<int*, MI355XSpace, MemoryTraits<Unmanaged>> order;
  int begin;
  KOKKOS_INLINE_FUNCTION void operator()(const int i) const {
    const int j = begin + i;
    const int b = op.bin(keys, j);
    order(offsets(b) + atomic_fetch_add(&fill(b), 1)) = j;
  }
};
template <class T>
struct is_bin_op_1d : std::false_type {};
template <class K>
struct is_bin_op_1d<BinOp1D<K>> : std::true_type {};

template <class Dst, class Keys>
struct BinKeyCopyF {
  Dst dst;
  Keys keys;
  int begin;
  KOKKOS_INLINE_FUNCTION void operator()(const int i) const { dst(i) = keys(begin + i); }
};
struct BinShiftF {
  View<int*, MI355XSpace, MemoryTraits<Unmanaged>> order;
  int begin;
  KOKKOS_INLINE_FUNCTION void operator()(const int i) const { order(i) += begin; }
};

// ---- BinOp1D order by quantised keys
// A key's bin is the whole part of x = mul * (key - min), and x never
// decreases as the key grows, so floor(x * 2^frac) orders keys as they are,
// up to keys that share a cell of 1 / 2^frac bins, and its upper bits are the
// bin.  Four 8-bit passes over such 32-bit codes replace the eight of the
// float64 keys; BinRunsF then finds runs of one code whose keys are not in
// order and BinRunSortF orders them by the keys.
//
// flags: [0] number of runs listed, [1] whether some key falls in no bin, [2]
// whether a run is too long; the last two send the call to the sort of the
// keys.
constexpr int kBinRunMax = 64;
template <class Keys>
struct BinQuantiseF {
  Keys keys;
  double mul, min, scale, bins;
  uint32_t* code;
  uint32_t* flags;
  int begin;
  KOKKOS_INLINE_FUNCTION void operator()(const int i) const {
    const double x = mul * (static_cast<double>(keys(begin + i)) - min);
    const bool in  = x >= 0.0 && x < bins;  // false for NaN
    if (!in) flags[1] = 1;
    code[i] = in ? static_cast<uint32_t>(x * scale) : 0u;
  }
};
template <class Keys>
struct BinRunsF {
  Keys keys;
  const uint32_t* code;  // sorted
  const uint32_t* order;
  uint32_t* flags;
  uint32_t* runs;
  int begin, n;
  KOKKOS_INLINE_FUNCTION bool descends(int i) const {
    return keys(begin + int(order[i])) < keys(begin + int(order[i - 1]));
  }
  KOKKOS_INLINE_FUNCTION void operator()(const int i) const {
    if (i == 0 || code[i] != code[i - 1] || !descends(i)) return;
    int first = i - 1;  // the run's first descent lists it
    while (first > 0 && code[first - 1] == code[i]) {
      if (i - first >= kBinRunMax) {
        flags[2] = 1;
        return;
      }
      if (descends(first)) return;
      --first;
    }
    runs[atomic_fetch_add(&flags[0], 1u)] = uint32_t(first);
  }
};
template <class Keys>
struct BinRunSortF {
  Keys keys;
  const uint32_t* code;
  uint32_t* order;
  uint32_t* flags;
  const uint32_t* runs;
  int begin, n;
  KOKKOS_INLINE_FUNCTION void operator()(const int start) const {
    const int listed = int(flags[0]);
    for (int r = start; r < listed; r += kRunLanes) {
      const int lo = int(runs[r]);
      for (int k = lo + 1; k < n && code[k] == code[lo]; ++k) {
        if (k - lo >= kBinRunMax) {
          flags[2] = 1;
          break;
        }
        const uint32_t cur = order[k];
        int j              = k - 1;
        while (j >= lo && keys(begin + int(cur)) < keys(begin + int(order[j]))) {
          order[j + 1] = order[j];
          --j;
        }
        order[j + 1] = cur;
      }
    }
  }
  static constexpr int kRunLanes = 1 << 16;
};
// Each bin's first position, that of the first sorted code that is not below
// it, and its count, from the next bin's, by two searches side by side.  Bin 0
// hands the flags to the host and clears them for the next call.
struct BinStartF {
  const uint32_t* code;
  View<int*, MI355XSpace, MemoryTraits<Unmanaged>> offsets, count;
  int n, frac, bins;
  uint32_t* flags;
  uint32_t* host;
  KOKKOS_INLINE_FUNCTION void operator()(const int b) const {
    const uint32_t want = uint32_t(b) << frac, next = uint32_t(b + 1) << frac;
    int lo = 0, hi = n, lo1 = 0, hi1 = n;
    while (lo < hi || lo1 < hi1) {
      const int mid = lo + (hi - lo) / 2, mid1 = lo1 + (hi1 - lo1) / 2;
      const uint32_t c = code[mid < n ? mid : n - 1], c1 = code[mid1 < n ? mid1 : n - 1];
      if (lo < hi) (c < want ? lo : hi) = c < want ? mid + 1 : mid;
      if (lo1 < hi1) (c1 < next ? lo1 : hi1) = c1 < next ? mid1 + 1 : mid1;
    }
    offsets(b) = lo;
    count(b)   = (b + 1 < bins ? lo1 : n) - lo;  // the last bin's next may not fit 32 bits
    if (b == 0) {
      for (int k = 1; k < 3; ++k) host[k] = flags[k];
      for (int k = 0; k < 3; ++k) flags[k] = 0;
    }
  }
};
struct BinZeroF {
  View<int*, MI355XSpace, MemoryTraits<Unmanaged>> order, count, offsets;
  KOKKOS_INLINE_FUNCTION void operator()(const size_t i) const {
    if (i < order.extent(0)) order(i) = 0;
    if (i < count.extent(0)) count(i) = offsets(i) = 0;
  }
};

// Device scratch of BinSort, kept between calls and grown on demand: held by
// its mutex until the stream has run what uses it; freed by Kokkos::finalize.
// `flags` are the ordering's, all zero between calls unless one was cut off by
// an error (clear is false then), `host` its pinned copy.
struct BinWorkspace {
  std::mutex mtx;
  void* buf       = nullptr;
  size_t bytes    = 0;
  bool hooked     = false;
  void* flags     = nullptr;
  uint32_t* host  = nullptr;
  bool clear      = false;
  void* space(size_t need);
};
// Values of a sorter go through the kept scratch up to this size, larger ones
// through a copy of their own: rows can be of any size, and the scratch stays.
constexpr size_t kBinRowsKept = size_t(256) << 20;
inline BinWorkspace& bin_workspace() {
  static BinWorkspace w;
  return w;
}
inline void bin_workspace_release() {
  BinWorkspace& w = bin_workspace();
  std::lock_guard<std::mutex> lock(w.mtx);
  if (w.buf) KKMX_SAFE_CALL(mx_free(w.buf, nullptr));
  if (w.flags) KKMX_SAFE_CALL(mx_free(w.flags, nullptr));
  if (w.host) KKMX_SAFE_CALL(mx_host_free(w.host));
  w.buf    = nullptr;
  w.flags  = nullptr;
  w.host   = nullptr;
  w.bytes  = 0;
  w.clear  = false;
  w.hooked = false;
}
inline void* BinWorkspace::space(size_t need) {
  if (bytes < need) {
    if (buf) KKMX_SAFE_CALL(mx_free(buf, nullptr));
    buf   = nullptr;
    bytes = 0;
    KKMX_SAFE_CALL(mx_malloc(&buf, need, nullptr));
    bytes = need;
  }
  if (!hooked) {
    push_finalize_hook(&bin_workspace_release);
    hooked = true;
  }
  return buf;
}

// The permutation of "by bin, then by key, equal keys in index order", bin
// counts and offsets, for len > 0.  False, with nothing defined, when some key
// falls in no bin.  Where more than kBinRunMax keys that are not in order
// share a code (keys crowded into a few cells), the keys themselves are
// sorted, which a BinOp1D never decreasing in the key makes the same order.
template <class Keys, class Op>
bool bin_order_by_code(const MI355X& exec, const Keys& keys, const Op& op, int begin, int len, int bins, int* order,
                       int* count, int* offsets) {
  using T = typename Keys::non_const_value_type;
  if (!(op.mul_ > 0.0) || bins < 1) return false;  // also a range that is no number
  int frac = 31;
  while (frac > 0 && (uint64_t(bins) << frac) > (uint64_t(1) << 32)) --frac;
  BinWorkspace& ws = bin_workspace();
  std::lock_guard<std::mutex> lock(ws.mtx);
  const bool few          = len <= kRadixMerged;
  const size_t code_bytes = radix_round(size_t(len) * 4);
  char* base              = static_cast<char*>(ws.space(2 * code_bytes + (few ? kRadixMergeBytes : 0)));
  uint32_t* code          = reinterpret_cast<uint32_t*>(base);
  uint32_t* runs          = reinterpret_cast<uint32_t*>(base + code_bytes);
  uint32_t* perm          = reinterpret_cast<uint32_t*>(order);
  if (!ws.flags) KKMX_SAFE_CALL(mx_malloc(&ws.flags, 64, nullptr));
  if (!ws.host) {
    void* h = nullptr;
    KKMX_SAFE_CALL(mx_host_alloc(&h, 64));
    ws.host = static_cast<uint32_t*>(h);
  }
  uint32_t* flags = static_cast<uint32_t*>(ws.flags);
  if (!ws.clear) clear_words_async(flags, 16, exec.stream());
  ws.clear = false;
  parallel_for("Kokkos::Sort::BinQuantise", RangePolicy<MI355X>(exec, 0, len),
               BinQuantiseF<Keys>{keys, op.mul_, op.min_, double(uint64_t(1) << frac), double(bins), code, flags, begin});
  if (few) radix_sort_few<uint32_t, uint32_t, true>(exec, code, len, perm, base + 2 * code_bytes);
  else radix_sort<uint32_t, uint32_t, true>(exec, code, int64_t(len), perm);
  parallel_for("Kokkos::Sort::BinRuns", RangePolicy<MI355X>(exec, 0, len),
               BinRunsF<Keys>{keys, code, perm, flags, runs, begin, len});
  const int lanes = len < BinRunSortF<Keys>::kRunLanes ? len : BinRunSortF<Keys>::kRunLanes;
  parallel_for("Kokkos::Sort::BinRunSort", RangePolicy<MI355X>(exec, 0, lanes),
               BinRunSortF<Keys>{keys, code, perm, flags, runs, begin, len});
  using U = View<int*, MI355XSpace, MemoryTraits<Unmanaged>>;
  parallel_for("Kokkos::Sort::BinStart", RangePolicy<MI355X>(exec, 0, bins),
               BinStartF{code, U(offsets, size_t(bins)), U(count, size_t(bins)), len, frac, bins, flags, ws.host});
  exec.fence("Kokkos::BinSort: keys in order");
  ws.clear                     = true;
  const volatile uint32_t* got = ws.host;
  if (got[1]) return false;
  if (got[2]) {
    View<T*, MI355XSpace> copy(view_alloc(WithoutInitializing, std::string("Kokkos::BinSort::key_copy")), size_t(len));
    parallel_for("Kokkos::Sort::BinKeyCopy", RangePolicy<MI355X>(exec, 0, len),
                 BinKeyCopyF<View<T*, MI355XSpace>, Keys>{copy, keys, begin});
    radix_sort<T, uint32_t, true>(exec, copy.data(), int64_t(len), perm);
  }
  return true;
}

// Insertion sort of one bin's indices by one thread, as the reference does on
// devices (quadratic in the bin size: meant for the small bins BinSort is
// used with); equal keys keep index order, so the result does not depend on
// the order the binning atomics ran in.
template <class Keys, class Op>
struct BinSortWithinF {
  Keys keys;
  Op op;
  View<const int*, MI355XSpace, MemoryTraits<Unmanaged>> count;
  View<const int*, MI355XSpace, MemoryTraits<Unmanaged>> offsets;
  View<int*, MI355XSpace, MemoryTraits<Unmanaged>> order;
  KOKKOS_INLINE_FUNCTION void operator()(const int b) const {
    const int lo = offsets(b), hi = lo + count(b);
    for (int k = lo + 1; k < hi; ++k) {
      int cur = order(k);
      int j   = k - 1;
      while (j >= lo) {
        int prev       = order(j);
        const bool before = op(keys, cur, prev) || (!op(keys, prev, cur) && cur < prev);
        if (!before) break;
        order(j + 1) = prev;
        --j;
      }
      order(j + 1) = cur;
    }
  }
};
template <class Dst, class Src>
struct PermuteRowsF {
  Dst dst;  // rows [0, len)
  Src src;
  View<const int*, MI355XSpace, MemoryTraits<Unmanaged>> order;
  int shift;  // values index = order(i) + shift
  KOKKOS_INLINE_FUNCTION void operator()(const int i) const {
    const int s = order(i) + shift;
    if constexpr (Dst::rank == 1) {
      dst(i) = src(s);
    } else {
      for (size_t c = 0; c < dst.extent(1); ++c) dst(i, c) = src(s, c);
    }
  }
};
template <class Dst, class Src>
struct CopyRowsF {
  Dst dst;
  Src src;
  int begin;  // dst rows [begin, begin + len)
  KOKKOS_INLINE_FUNCTION void operator()(const int i) const {
    if constexpr (Dst::rank == 1) {
      dst(begin + i) = src(i);
    } else {
      for (size_t c = 0; c < dst.extent(1); ++c) dst(begin + i, c) = src(i, c);
    }
  }
};

}  // namespace Impl

// ------------------------------------------------------------------ sort helpers
namespace Impl {

template <class V>
constexpr bool radix_sortable() {
  using T = typename V::non_const_value_type;
  return V::rank == 1 && std::is_arithmetic<T>::value && !std::is_same<T, bool>::value &&
         (sizeof(T) == 4 || sizeof(T) == 8) && exec_can_access<MI355X, typename V::memory_space>::value;
}

template <class V, class Comp>
void host_sort(const V& view, size_t begin, size_t end, Comp comp) {
  using T = typename V::non_const_value_type;
  const size_t n = end - begin;
  std::vector<T> h(n);
  if constexpr (exec_can_access<Serial, typename V::memory_space>::value) {
    for (size_t i = 0; i < n; ++i) h[i] = view(begin + i);
    std::sort(h.begin(), h.end(), comp);
    for (size_t i = 0; i < n; ++i) view(begin + i) = h[i];
  } else {
    static_assert(V::rank == 1, "Kokkos::sort sorts rank-1 Views");
    Kokkos::fence("Kokkos::sort: host fallback");
    if (view.span_is_contiguous()) {
      KKMX_SAFE_CALL(mx_memcpy(h.data(), view.data() + begin, n * sizeof(T)));
      std::sort(h.begin(), h.end(), comp);
      KKMX_SAFE_CALL(mx_memcpy(view.data() + begin, h.data(), n * sizeof(T)));
    } else {
      auto m = create_mirror_view_and_copy(HostSpace(), view);
      for (size_t i = 0; i < n; ++i) h[i] = m(begin + i);
      std::sort(h.begin(), h.end(), comp);
      for (size_t i = 0; i < n; ++i) m(begin + i) = h[i];
      deep_copy(view, m);
    }
  }
}

}  // namespace Impl

// ------------------------------------------------------------------ BinSort
template <class KeyViewType, class BinSortOp, class Space = typename KeyViewType::device_type,
          class SizeType = typename KeyViewType::size_type>
class BinSort {
 public:
  using exec_space       = MI355X;
  using offset_type      = View<int*, MI355XSpace>;
  using bin_count_type   = View<const int*, MI355XSpace>;
  using const_key_view_type = typename KeyViewType::const_type;

  BinSort() = delete;
  template <class ExecutionSpace>
  BinSort(const ExecutionSpace& exec, const_key_view_type keys_, int range_begin_, int range_end_, BinSortOp bin_op_,
          bool sort_within_bins_ = false)
      : keys(keys_),
        range_begin(range_begin_),
        range_end(range_end_),
        bin_op(bin_op_),
        sort_within_bins(sort_within_bins_) {
    static_assert(std::is_same<ExecutionSpace, MI355X>::value, "BinSort runs on the MI355X execution space");
    if (range_begin > range_end) Kokkos::abort("BinSort: range_begin > range_end");
    const size_t len = size_t(range_end - range_begin), bins = size_t(bin_op.max_bins());
    sort_order  = offset_type(view_alloc(WithoutInitializing, std::string("Kokkos::BinSort::sort_order")), len);
    bin_count   = View<int*, MI355XSpace>(view_alloc(WithoutInitializing, std::string("Kokkos::BinSort::bin_count")), bins);
    bin_offsets = offset_type(view_alloc(WithoutInitializing, std::string("Kokkos::BinSort::bin_offsets")), bins);
    // made here and not where it is used, so that create_permute_vector can be
    // captured; a radix sort cannot, and its calls hardly ever need it
    if (!(by_code && sort_within_bins && len > 0))
      bin_fill = View<int*, MI355XSpace>(view_alloc(WithoutInitializing, std::string("Kokkos::BinSort::bin_fill")), bins);
    // one launch and one wait for all three
    using U = View<int*, MI355XSpace, MemoryTraits<Unmanaged>>;
    parallel_for("Kokkos::Sort::BinZero", RangePolicy<MI355X, IndexType<size_t>>(exec, 0, len > bins ? len : bins),
                 Impl::BinZeroF{U(sort_order.data(), len), U(bin_count.data(), bins), U(bin_offsets.data(), bins)});
    exec.fence("Kokkos::BinSort: Views set to zero");
  }
  BinSort(const_key_view_type keys_, int range_begin_, int range_end_, BinSortOp bin_op_, bool sort_within_bins_ = false)
      : BinSort(exec_space{}, keys_, range_begin_, range_end_, bin_op_, sort_within_bins_) {}
  template <class ExecutionSpace>
  BinSort(const ExecutionSpace& exec, const_key_view_type keys_, BinSortOp bin_op_, bool sort_within_bins_ = false)
      : BinSort(exec, keys_, 0, int(keys_.extent(0)), bin_op_, sort_within_bins_) {}
  BinSort(const_key_view_type keys_, BinSortOp bin_op_, bool sort_within_bins_ = false)
      : BinSort(exec_space{}, keys_, bin_op_, sort_within_bins_) {}

  // Counts, offsets and the permutation; call again when the keys change.
  template <class ExecutionSpace>
  void create_permute_vector(const ExecutionSpace& exec) {
    using U        = View<int*, MI355XSpace, MemoryTraits<Unmanaged>>;
    using CU       = View<const int*, MI355XSpace, MemoryTraits<Unmanaged>>;
    const int len  = range_end - range_begin;
    const int bins = bin_op.max_bins();
    U cnt(bin_count.data(), size_t(bins));
    U off(bin_offsets.data(), size_t(bins)), order(sort_order.data(), size_t(len));
    if constexpr (by_code) {
      if (sort_within_bins && len > 0 &&
          Impl::bin_order_by_code(exec, keys, bin_op, range_begin, len, bins, order.data(), cnt.data(), off.data())) {
        if (range_begin != 0)
          parallel_for("Kokkos::Sort::BinShift", RangePolicy<MI355X>(exec, 0, len), Impl::BinShiftF{order, range_begin});
        return;
      }
    }
    if (bin_fill.extent(0) != size_t(bins)) bin_fill = View<int*, MI355XSpace>("Kokkos::BinSort::bin_fill", size_t(bins));
    U fill(bin_fill.data(), size_t(bins));
    deep_copy(exec, bin_count, 0);
    deep_copy(exec, bin_fill, 0);
    parallel_for("Kokkos::Sort::BinCount", RangePolicy<MI355X>(exec, 0, len),
                 Impl::BinCountF<const_key_view_type, BinSortOp>{keys, bin_op, cnt, range_begin});
    parallel_scan("Kokkos::Sort::BinOffset", RangePolicy<MI355X>(exec, 0, bins), Impl::BinOffsetF{CU(cnt), off});
    if constexpr (by_code) {
      // BinOp1D's bin never decreases as the key grows, so "by bin, then by
      // key, equal keys in index order" is the stable order of the keys: the
      // permutation of a radix sort of (key, position) pairs
      if (sort_within_bins && len > 0) {
        using T = typename KeyViewType::non_const_value_type;
        View<T*, MI355XSpace> copy(view_alloc(WithoutInitializing, std::string("Kokkos::BinSort::key_copy")),
                                   size_t(len));
        parallel_for("Kokkos::Sort::BinKeyCopy", RangePolicy<MI355X>(exec, 0, len),
                     Impl::BinKeyCopyF<View<T*, MI355XSpace>, const_key_view_type>{copy, keys, range_begin});
        Impl::radix_sort<T, uint32_t, true>(exec, copy.data(), int64_t(len),
                                            reinterpret_cast<uint32_t*>(sort_order.data()));
        if (range_begin != 0)
          parallel_for("Kokkos::Sort::BinShift", RangePolicy<MI355X>(exec, 0, len), Impl::BinShiftF{order, range_begin});
        return;
      }
    }
    parallel_for("Kokkos::Sort::BinBinning", RangePolicy<MI355X>(exec, 0, len),
                 Impl::BinPlaceF<const_key_view_type, BinSortOp>{keys, bin_op, fill, CU(off), order, range_begin});
    if (sort_within_bins)
      parallel_for("Kokkos::Sort::BinSort", RangePolicy<MI355X>(exec, 0, bins),
                   Impl::BinSortWithinF<const_key_view_type, BinSortOp>{keys, bin_op, CU(cnt), CU(off), order});
  }
  void create_permute_vector() {
    Kokkos::fence("Kokkos::BinSort::create_permute_vector: before");
    exec_space e{};
    create_permute_vector(e);
    e.fence("Kokkos::BinSort::create_permute_vector: after");
  }

  // values(range_begin + i) = values(sort_order(i) + values_range_begin - range_begin)
  template <class ExecutionSpace, class ValuesViewType>
  void sort(const ExecutionSpace& exec, const ValuesViewType& values, int values_range_begin,
            int values_range_end) const {
    if (values.extent(0) == 0) return;
    const int len = range_end - range_begin;
    if (values_range_end - values_range_begin != len)
      Kokkos::abort("BinSort::sort: values range length != permutation vector length");
    View<const int*, MI355XSpace, MemoryTraits<Unmanaged>> order(sort_order.data(), size_t(len));
    using W = typename ValuesViewType::non_const_value_type;
    if constexpr (ValuesViewType::rank == 1 && std::is_trivially_copyable<W>::value) {
      // through the kept scratch, which is free again once the stream is done
      using Rows               = View<W*, MI355XSpace, MemoryTraits<Unmanaged>>;
      const size_t need        = size_t(len) * sizeof(W);
      Impl::BinWorkspace& ws   = Impl::bin_workspace();
      std::lock_guard<std::mutex> lock(ws.mtx);
      if (need <= Impl::kBinRowsKept || need <= ws.bytes) {
        Rows rows(static_cast<W*>(ws.space(need)), size_t(len));
        parallel_for("Kokkos::Sort::CopyPermute", RangePolicy<MI355X>(exec, 0, len),
                     Impl::PermuteRowsF<Rows, ValuesViewType>{rows, values, order, values_range_begin - range_begin});
        parallel_for("Kokkos::Sort::Copy", RangePolicy<MI355X>(exec, 0, len),
                     Impl::CopyRowsF<ValuesViewType, Rows>{values, rows, range_begin});
        exec.fence("Kokkos::BinSort::sort: values in place");
        return;
      }
    }
    using Tmp = View<typename ValuesViewType::non_const_data_type, typename ValuesViewType::array_layout, MI355XSpace>;
    Tmp tmp(std::string("Kokkos::SortImpl::BinSortFunctor::sorted_values"), size_t(len),
            ValuesViewType::rank > 1 ? values.extent(1) : ~size_t(0));  // ~0: no extent
    parallel_for("Kokkos::Sort::CopyPermute", RangePolicy<MI355X>(exec, 0, len),
                 Impl::PermuteRowsF<Tmp, ValuesViewType>{tmp, values, order, values_range_begin - range_begin});
    parallel_for("Kokkos::Sort::Copy", RangePolicy<MI355X>(exec, 0, len),
                 Impl::CopyRowsF<ValuesViewType, Tmp>{values, tmp, range_begin});
  }
  template <class ValuesViewType>
  void sort(const ValuesViewType& values, int values_range_begin, int values_range_end) const {
    Kokkos::fence("Kokkos::BinSort::sort: before");
    exec_space exec;
    sort(exec, values, values_range_begin, values_range_end);
    exec.fence("Kokkos::BinSort::sort: after");
  }
  template <class ExecutionSpace, class ValuesViewType, class = std::enable_if_t<is_execution_space<ExecutionSpace>::value>>
  void sort(const ExecutionSpace& exec, const ValuesViewType& values) const {
    sort(exec, values, 0, range_end - range_begin);
  }
  template <class ValuesViewType>
  void sort(const ValuesViewType& values) const {
    sort(values, 0, range_end - range_begin);
  }

  offset_type get_permute_vector() const { return sort_order; }
  offset_type get_bin_offsets() const { return bin_offsets; }
  bin_count_type get_bin_count() const { return bin_count; }

 private:
  // within bins, the ordering is a radix sort
  static constexpr bool by_code =
      Impl::is_bin_op_1d<BinSortOp>::value && KeyViewType::rank == 1 && Impl::radix_sortable<KeyViewType>();
  const_key_view_type keys;
  int range_begin = 0, range_end = 0;
  BinSortOp bin_op;
  bool sort_within_bins = false;
  offset_type sort_order;
  View<int*, MI355XSpace> bin_count, bin_fill;
  offset_type bin_offsets;
};

// ------------------------------------------------------------------ sort
template <class ExecutionSpace, class DataType, class... Properties,
          class = std::enable_if_t<is_execution_space<ExecutionSpace>::value>>
void sort(const ExecutionSpace& exec, const View<DataType, Properties...>& view) {
  using V = View<DataType, Properties...>;
  using T = typename V::non_const_value_type;
  static_assert(V::rank == 1, "Kokkos::sort sorts rank-1 Views");
  if (view.extent(0) < 2) return;
  if constexpr (Impl::radix_sortable<V>() && std::is_same<ExecutionSpace, MI355X>::value) {
    if (view.span_is_contiguous()) {
      Impl::radix_sort<T>(exec, view.data(), int64_t(view.extent(0)));
    } else {
      // strided keys: gather into a contiguous copy, sort it, scatter back
      View<T*, MI355XSpace> packed(view_alloc(WithoutInitializing, std::string("Kokkos::sort::packed")),
                                   view.extent(0));
      deep_copy(exec, packed, view);
      Impl::radix_sort<T>(exec, packed.data(), int64_t(packed.extent(0)));
      deep_copy(exec, view, packed);
      exec.fence("Kokkos::sort: strided keys written back");
    }
    return;
  }
  exec.fence();
  Impl::host_sort(view, 0, view.extent(0), std::less<T>());
}
template <class DataType, class... Properties>
void sort(const View<DataType, Properties...>& view) {
  Kokkos::fence("Kokkos::sort: before");
  sort(MI355X(), view);
  Kokkos::fence("Kokkos::sort: after");
}
template <class ExecutionSpace, class Comparator, class DataType, class... Properties,
          class = std::enable_if_t<is_execution_space<ExecutionSpace>::value>>
void sort(const ExecutionSpace& exec, const View<DataType, Properties...>& view, const Comparator& comp) {
  exec.fence();
  Impl::host_sort(view, 0, view.extent(0), comp);
}
template <class Comparator, class DataType, class... Properties,
          class = std::enable_if_t<!is_execution_space<Comparator>::value>>
void sort(const View<DataType, Properties...>& view, const Comparator& comp) {
  Kokkos::fence("Kokkos::sort: before");
  Impl::host_sort(view, 0, view.extent(0), comp);
}
template <class ExecutionSpace, class ViewType, class = std::enable_if_t<is_execution_space<ExecutionSpace>::value>>
void sort(const ExecutionSpace& exec, ViewType view, size_t begin, size_t end) {
  using T = typename ViewType::non_const_value_type;
  if (end <= begin + 1) return;
  if constexpr (Impl::radix_sortable<ViewType>() && std::is_same<ExecutionSpace, MI355X>::value) {
    if (view.span_is_contiguous()) {
      Impl::radix_sort<T>(exec, view.data() + begin, int64_t(end - begin));
      return;
    }
    // strided keys: the same gather / sort / scatter over [begin, end)
    View<T*, MI355XSpace> packed(view_alloc(WithoutInitializing, std::string("Kokkos::sort::packed")), end - begin);
    auto window = subview(view, std::make_pair(begin, end));
    deep_copy(exec, packed, window);
    Impl::radix_sort<T>(exec, packed.data(), int64_t(packed.extent(0)));
    deep_copy(exec, window, packed);
    exec.fence("Kokkos::sort: strided keys written back");
    return;
  }
  exec.fence();
  Impl::host_sort(view, begin, end, std::less<T>());
}
template <class ViewType>
void sort(ViewType view, size_t begin, size_t end) {
  Kokkos::fence("Kokkos::sort: before");
  sort(MI355X(), view, begin, end);
  Kokkos::fence("Kokkos::sort: after");
}

// ------------------------------------------------------------------ sort_by_key
// algorithms/src/sorting/Kokkos_SortByKeyPublicAPI.hpp:27-108 and
// impl/Kokkos_SortByKeyImpl.hpp:98-109 (admissible Views), 262-324
// (permutation fallback).  Keys that the radix sort takes are sorted on the
// device with the values riding along as radix payload (contiguous values of
// 4 or 8 bytes) or as (key, position) pairs whose permutation then gathers
// the values; either way equal keys keep their input order, as with the
// rocThrust path (impl/Kokkos_SortByKeyImpl.hpp:145-158).  A comparator, or keys
// the radix sort does not take, sort a permutation on the host with
// std::stable_sort.
namespace Impl {

template <class V>
constexpr bool sort_by_key_admissible() {
  using L = typename V::array_layout;
  return is_view<V>::value && V::rank == 1 &&
         (std::is_same<L, LayoutLeft>::value || std::is_same<L, LayoutRight>::value ||
          std::is_same<L, LayoutStride>::value);
}

template <class Dst, class Src>
struct SortByKeyCopyF {
  Dst dst;
  Src src;
  KOKKOS_INLINE_FUNCTION void operator()(const int64_t i) const { dst(i) = src(i); }
};
template <class Dst, class Src, class P>
struct SortByKeyGatherF {
  Dst dst;
  Src src;
  P perm;
  KOKKOS_INLINE_FUNCTION void operator()(const int64_t i) const { dst(i) = src(perm(i)); }
};

// view(i) = view(perm(i)) for every i, through a device copy of view.
template <class VV, class P>
void apply_permutation(const MI355X& exec, const P& perm, const VV& view) {
  using T         = typename VV::non_const_value_type;
  const int64_t n = int64_t(view.extent(0));
  View<T*, MI355XSpace> copy(view_alloc(WithoutInitializing, std::string("Kokkos::sort_by_key::permute_copy")),
                             size_t(n));
  parallel_for("Kokkos::sort_by_key::copy", RangePolicy<MI355X, IndexType<int64_t>>(exec, 0, n),
               SortByKeyCopyF<decltype(copy), VV>{copy, view});
  parallel_for("Kokkos::sort_by_key::gather", RangePolicy<MI355X, IndexType<int64_t>>(exec, 0, n),
               SortByKeyGatherF<VV, decltype(copy), P>{view, copy, perm});
  exec.fence("Kokkos::sort_by_key: permuted");
}

template <class KV, class VV, class Comp>
void sort_by_key_host(const KV& keys, const VV& values, Comp comp) {
  const size_t n = keys.extent(0);
  auto hk        = create_mirror_view_and_copy(HostSpace(), keys);
  auto hv        = create_mirror_view_and_copy(HostSpace(), values);
  std::vector<uint32_t> idx(n);
  for (size_t i = 0; i < n; ++i) idx[i] = uint32_t(i);
  std::stable_sort(idx.begin(), idx.end(), [&](uint32_t a, uint32_t b) { return comp(hk(a), hk(b)); });
  std::vector<typename KV::non_const_value_type> k(n);
  std::vector<typename VV::non_const_value_type> v(n);
  for (size_t i = 0; i < n; ++i) {
    k[i] = hk(idx[i]);
    v[i] = hv(idx[i]);
  }
  for (size_t i = 0; i < n; ++i) {
    hk(i) = k[i];
    hv(i) = v[i];
  }
  deep_copy(keys, hk);
  deep_copy(values, hv);
}

template <class ExecutionSpace, class KV, class VV>
void check_sort_by_key(const KV& keys, const VV& values) {
  static_assert(sort_by_key_admissible<KV>() && sort_by_key_admissible<VV>(),
                "Kokkos::sort_by_key only accepts 1D values View with LayoutRight, LayoutLeft or LayoutStride.");
  static_assert(SpaceAccessibility<ExecutionSpace, typename KV::memory_space>::accessible,
                "Kokkos::sort: execution space instance is not able to access the memory space of the keys View "
                "argument!");
  static_assert(SpaceAccessibility<ExecutionSpace, typename VV::memory_space>::accessible,
                "Kokkos::sort: execution space instance is not able to access the memory space of the values View "
                "argument!");
  if (values.size() != keys.size())
    Kokkos::abort((std::string("values and keys extents must be the same. The values extent is ") +
                   std::to_string(values.size()) + ", and the keys extent is " + std::to_string(keys.size()) + ".")
                      .c_str());
}

}  // namespace Impl

namespace Experimental {

template <class ExecutionSpace, class KeysDataType, class... KeysProperties, class ValuesDataType,
          class... ValuesProperties>
void sort_by_key(const ExecutionSpace& exec, const View<KeysDataType, KeysProperties...>& keys,
                 const View<ValuesDataType, ValuesProperties...>& values) {
  using KV = View<KeysDataType, KeysProperties...>;
  using VV = View<ValuesDataType, ValuesProperties...>;
  using T  = typename KV::non_const_value_type;
  Kokkos::Impl::check_sort_by_key<ExecutionSpace>(keys, values);
  if (keys.extent(0) <= 1) return;
  if constexpr (Kokkos::Impl::radix_sortable<KV>() && std::is_same<ExecutionSpace, MI355X>::value) {
    if (keys.span_is_contiguous()) {
      using W = typename VV::non_const_value_type;
      if constexpr ((sizeof(W) == 4 || sizeof(W) == 8) && std::is_trivially_copyable<W>::value) {
        if (values.span_is_contiguous()) {
          // the values ride through the radix passes with their keys
          using PT = std::conditional_t<sizeof(W) == 4, uint32_t, uint64_t>;
          Kokkos::Impl::radix_sort<T, PT>(exec, keys.data(), int64_t(keys.extent(0)),
                                          reinterpret_cast<PT*>(values.data()));
          return;
        }
      }
      View<uint32_t*, MI355XSpace> perm(view_alloc(WithoutInitializing, std::string("Kokkos::sort_by_key::permute")),
                                        keys.extent(0));
      Kokkos::Impl::radix_sort<T, uint32_t, true>(exec, keys.data(), int64_t(keys.extent(0)), perm.data());
      Kokkos::Impl::apply_permutation(exec, perm, values);
      return;
    }
  }
  exec.fence("Kokkos::sort_by_key: before host sort");
  Kokkos::Impl::sort_by_key_host(keys, values, std::less<T>());
}

template <class ExecutionSpace, class ComparatorType, class KeysDataType, class... KeysProperties,
          class ValuesDataType, class... ValuesProperties>
void sort_by_key(const ExecutionSpace& exec, const View<KeysDataType, KeysProperties...>& keys,
                 const View<ValuesDataType, ValuesProperties...>& values, const ComparatorType& comparator) {
  Kokkos::Impl::check_sort_by_key<ExecutionSpace>(keys, values);
  if (keys.extent(0) <= 1) return;
  exec.fence("Kokkos::sort_by_key: before host sort");
  Kokkos::Impl::sort_by_key_host(keys, values, comparator);
}

}  // namespace Experimental

}  // namespace Kokkos

#endif
