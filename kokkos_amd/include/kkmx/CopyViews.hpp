// deep_copy, create_mirror, create_mirror_view, create_mirror_view_and_copy,
// realloc/resize.
//
// Reference: core/src/Kokkos_CopyViews.hpp:58-420 (ViewFill / ViewCopy are
// parallel_for kernels; whole-allocation copies of contiguous Views go to the
// runtime memcpy), core/src/HIP/Kokkos_HIP_DeepCopy.cpp:23-51.
// deep_copy without an execution space fences before and after, as in the
// reference; deep_copy(exec, ...) is ordered on exec's stream only.
#ifndef KKMX_COPY_VIEWS_HPP
#define KKMX_COPY_VIEWS_HPP

#include <kkmx/Parallel.hpp>

namespace Kokkos {
namespace Impl {

template <class ViewT>
struct FillFunctor {
  using value_type = typename ViewT::non_const_value_type;
  typename ViewT::value_type* ptr;
  value_type val;
  KOKKOS_INLINE_FUNCTION void operator()(const int64_t i) const { ptr[i] = val; }
};

// Contiguous copy of elements (8-byte words when sizes and alignment allow).
template <class T>
struct CopyElems {
  const T* src;
  T* dst;
  KOKKOS_INLINE_FUNCTION void operator()(const int64_t i) const { dst[i] = src[i]; }
};

// Index-space fill and copy, for Views whose span is not their index space
// (LayoutStride) or whose layouts differ: MDRange over the extents (rank
// 2-6) or a Range (rank 1); the functor receives the View indices directly.
template <class ViewT>
struct IndexFill {
  ViewT dst;
  typename ViewT::non_const_value_type val;
  template <class... I>
  KOKKOS_INLINE_FUNCTION void operator()(const I... i) const {
    dst(i...) = val;
  }
};
template <class DV, class SV>
struct IndexCopy {
  DV dst;
  SV src;
  template <class... I>
  KOKKOS_INLINE_FUNCTION void operator()(const I... i) const {
    dst(i...) = src(i...);
  }
};

// A layout of v's extents with no padding: a LayoutStride gets compact
// strides, last index fastest.  Staging buffers are allocated from it, so a
// single transfer of size() elements moves them whole.
template <class V>
typename V::array_layout compact_layout(const V& v) {
  typename V::array_layout l{};
  size_t s = 1;
  for (int r = int(V::rank) - 1; r >= 0; --r) {
    l.dimension[r] = v.extent(r);
    if constexpr (std::is_same<typename V::array_layout, LayoutStride>::value) l.stride[r] = s;
    s *= v.extent(r);
  }
  return l;
}

template <class DV, class SV>
struct ElementCopy {
  DV dst;
  SV src;
  KOKKOS_INLINE_FUNCTION void operator()(const int64_t i) const {
    // Rank-generic element copy through a flat index (LayoutRight order).
    size_t idx[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int64_t r     = i;
    for (int d = int(DV::rank) - 1; d >= 0; --d) {
      const size_t e = dst.extent(d);
      idx[d]         = static_cast<size_t>(r % static_cast<int64_t>(e));
      r /= static_cast<int64_t>(e);
    }
    if constexpr (DV::rank == 0) dst() = src();
    else if constexpr (DV::rank == 1) dst(idx[0]) = src(idx[0]);
    else if constexpr (DV::rank == 2) dst(idx[0], idx[1]) = src(idx[0], idx[1]);
    else if constexpr (DV::rank == 3) dst(idx[0], idx[1], idx[2]) = src(idx[0], idx[1], idx[2]);
    else if constexpr (DV::rank == 4) dst(idx[0], idx[1], idx[2], idx[3]) = src(idx[0], idx[1], idx[2], idx[3]);
    else if constexpr (DV::rank == 5)
      dst(idx[0], idx[1], idx[2], idx[3], idx[4]) = src(idx[0], idx[1], idx[2], idx[3], idx[4]);
    else if constexpr (DV::rank == 6)
      dst(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5]) = src(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5]);
    else if constexpr (DV::rank == 7)
      dst(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5], idx[6]) =
          src(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5], idx[6]);
    else
      dst(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5], idx[6], idx[7]) =
          src(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5], idx[6], idx[7]);
  }
};

// ViewCopy between LayoutLeft and LayoutRight (both contiguous, rank >= 2)
// as an LDS-tiled transpose on gfx950: each 512-lane workgroup moves a tile of
// (first index, last index) for one multi-index of the middle dimensions, 64
// long in the source's contiguous dimension and 64 or, for some shapes of 8-byte
// words, 32 (transpose_narrow) in the destination's.  It reads along the
// source's contiguous dimension and writes along the destination's, both
// coalesced; the tile sits in LDS with an odd row pitch so neither pass has
// bank conflicts.  Consecutive workgroups take consecutive tiles of the last
// index, and the destination is written with nontemporal stores (a copy's
// output is not read back by the copy).  512^3 doubles: 0.436 ms a call
// (kernel trace 0.437 on average, 0.429 at best), 0.447 with 64 x 64 tiles and
// 64-bit index arithmetic.  Variants back to back in one loop: 0.421 with 64 x 32
// tiles, 0.435 with 64 x 64 (0.449 with 64-bit arithmetic), 0.51-0.64 with 128 in
// either direction, 0.65 with the middle index fastest.
//   LayoutLeft  offset of (i, mid, k) = i + e0 * (midL + M * k)
//   LayoutRight offset of (i, mid, k) = (i * M + midR) * e_last + k
// midL / midR: the middle indices flattened left-first / right-first, M
// their product.
struct TransposeShape {
  int64_t e0, elast, M;
  uint32_t mid[4];  // extents of the middle dimensions (1 when absent)
  int nmid;
  uint32_t tiles0, tileslast;  // their product with M is below 2^31
  uint32_t first;              // tile of the launch's first workgroup
};
// Tiles of one launch: HIP takes fewer than 2^32 lanes along a grid dimension.
constexpr int64_t kTransposeTiles = int64_t(1) << 22;
// N: tile extent along the destination's contiguous dimension.
template <class W, bool SrcLeft, int N>
__global__ __launch_bounds__(512) void k_layout_transpose(W* __restrict__ dst, const W* __restrict__ src,
                                                          const TransposeShape sh) {
  __shared__ W tile[N][65];
  const uint32_t b  = sh.first + blockIdx.x;
  const uint32_t tk = b % sh.tileslast;
  const uint32_t t0 = (b / sh.tileslast) % sh.tiles0;
  uint32_t g        = b / (sh.tiles0 * sh.tileslast);  // middle multi-index, flattened left-first
  int64_t midL = g, midR = 0;
  {
    uint32_t idx[4] = {0, 0, 0, 0};
    for (int d = 0; d < sh.nmid; ++d) {
      idx[d] = g % sh.mid[d];
      g /= sh.mid[d];
    }
    for (int d = 0; d < sh.nmid; ++d) midR = midR * sh.mid[d] + idx[d];
  }
  // load along the source's contiguous dimension
  const int lane = threadIdx.x & 63, row = threadIdx.x >> 6;
  const int64_t i0 = int64_t(t0) * (SrcLeft ? 64 : N), k0 = int64_t(tk) * (SrcLeft ? N : 64);
#pragma unroll
  for (int r = 0; r < N / 8; ++r) {
    const int q = row + 8 * r;
    if (SrcLeft) {
      const int64_t i = i0 + lane, k = k0 + q;
      if (i < sh.e0 && k < sh.elast) tile[q][lane] = src[i + sh.e0 * (midL + sh.M * k)];
    } else {
      const int64_t k = k0 + lane, i = i0 + q;
      if (i < sh.e0 && k < sh.elast) tile[q][lane] = src[(i * sh.M + midR) * sh.elast + k];
    }
  }
  __syncthreads();
  // store along the destination's contiguous dimension
  const int near = threadIdx.x % N, far = threadIdx.x / N;
#pragma unroll
  for (int r = 0; r < N / 8; ++r) {
    const int q = far + 512 / N * r;
    if (SrcLeft) {  // destination LayoutRight: k fastest; tile[k_local][i_local]
      const int64_t k = k0 + near, i = i0 + q;
      if (i < sh.e0 && k < sh.elast) __builtin_nontemporal_store(tile[near][q], &dst[(i * sh.M + midR) * sh.elast + k]);
    } else {  // destination LayoutLeft: i fastest; tile[i_local][k_local]
      const int64_t i = i0 + near, k = k0 + q;
      if (i < sh.e0 && k < sh.elast) __builtin_nontemporal_store(tile[near][q], &dst[i + sh.e0 * (midL + sh.M * k)]);
    }
  }
}
template <class T>
using transpose_word_t =
    std::conditional_t<sizeof(T) == 8, uint64_t,
                       std::conditional_t<sizeof(T) == 4, uint32_t, std::conditional_t<sizeof(T) == 2, uint16_t, uint8_t>>>;

// Whether 8-byte words take 64 x 32 tiles, which leave room for twice the
// workgroups on a CU but write rows of half the length.  `across` is the source's
// contiguous extent, `along` the destination's, `words` all of the copy.  Below 2^20
// words the smaller tiles reach more CUs: 0.85-1.05 of the time of 64 x 64 ones, from
// 2^20 to 2^21 0.9-1.1 with a middle above 1.  Of larger copies, to 32 M words:
//  * Half as long tiles are not twice as many where the last of them is at most
//    half full: 0.81-1.0 up to 32 along (1.0-1.07, and 1.25 at 17 by 48, for large
//    copies with rows that start within 64 bytes), 0.6-0.97 at 72 to 96, 0.74-1.03
//    at 200 to 224, 0.9-1.03 at 136 to 160 and from 264 on; but 1.04-1.2 there for
//    narrow sources, and 1.0-1.3 for rows that start within 64 bytes (65, 130).
//  * Otherwise the rows of a tile count: 1.1-1.7 at 33 to 48, 1.0-1.2 at 100, 112
//    and 300; even at 64, 128 and 256 (1.04-1.2 for narrow sources) and from 512 on
//    0.97 at 512^3.
inline bool transpose_narrow(int64_t across, int64_t along, int64_t words) {
  if (words < (int64_t(1) << 20) || along <= 32) return true;
  if (along % 8 != 0) return false;
  const int64_t last = along % 64;
  if (last == 0) return along >= 512 && across >= 64;
  return last <= 32 && (along < 128 || across >= 48);
}

// Launches the transpose when it applies (Left <-> Right, contiguous, rank
// 2-6, trivially copyable elements of 1-8 bytes, first and last extents of
// at least 16); returns false otherwise.
template <class DV, class SV>
bool layout_transpose(const MI355X& exec, const DV& dst, const SV& src) {
  using T            = typename DV::non_const_value_type;
  using DL           = typename DV::array_layout;
  using SL           = typename SV::array_layout;
  constexpr bool lr  = std::is_same<DL, LayoutRight>::value && std::is_same<SL, LayoutLeft>::value;
  constexpr bool rl  = std::is_same<DL, LayoutLeft>::value && std::is_same<SL, LayoutRight>::value;
  constexpr unsigned R = DV::rank;
  if constexpr (!(lr || rl) || R < 2 || R > 6 || !std::is_trivially_copyable<T>::value ||
                !(sizeof(T) == 1 || sizeof(T) == 2 || sizeof(T) == 4 || sizeof(T) == 8)) {
    return false;
  } else {
    if (!dst.span_is_contiguous() || !src.span_is_contiguous()) return false;
    TransposeShape sh{};
    sh.e0    = int64_t(dst.extent(0));
    sh.elast = int64_t(dst.extent(R - 1));
    if (sh.e0 < 16 || sh.elast < 16) return false;
    sh.M    = 1;
    sh.nmid = int(R) - 2;
    for (int d = 0; d < 4; ++d) sh.mid[d] = 1;
    for (int d = 0; d < sh.nmid; ++d) {
      sh.M *= int64_t(dst.extent(d + 1));
      sh.mid[d] = uint32_t(dst.extent(d + 1));
    }
    if (sh.M == 0) return true;
    using W              = transpose_word_t<T>;
    const int64_t across = lr ? sh.e0 : sh.elast, along = lr ? sh.elast : sh.e0;
    const int N          = sizeof(W) == 8 && transpose_narrow(across, along, int64_t(dst.span())) ? 32 : 64;
    const int64_t tiles0 = lr ? (sh.e0 + 63) / 64 : (sh.e0 + N - 1) / N;
    const int64_t tileslast = lr ? (sh.elast + N - 1) / N : (sh.elast + 63) / 64;
    if (tiles0 > 0x7fffffff || tileslast > 0x7fffffff / tiles0 || sh.M > 0x7fffffff / (tiles0 * tileslast)) return false;
    const int64_t blocks = tiles0 * tileslast * sh.M;
    sh.tiles0            = uint32_t(tiles0);
    sh.tileslast         = uint32_t(tileslast);
    W* d                 = reinterpret_cast<W*>(dst.data());
    const W* s_          = reinterpret_cast<const W*>(src.data());
    const void* k        = reinterpret_cast<const void*>(&k_layout_transpose<W, lr, 64>);
    if constexpr (sizeof(W) == 8)
      if (N == 32) k = reinterpret_cast<const void*>(&k_layout_transpose<W, lr, 32>);
    for (int64_t done = 0; done < blocks; done += kTransposeTiles) {
      sh.first            = uint32_t(done);
      const int64_t tiles = blocks - done < kTransposeTiles ? blocks - done : kTransposeTiles;
      mx_launch_kernel(k, static_cast<unsigned>(tiles), 512, 0, exec.stream(), d, s_, sh);
    }
    return true;
  }
}

// Runs f over the index space of v on exec: a Range for rank 1, an MDRange
// (iterating in v's layout order, so consecutive lanes touch consecutive
// addresses of v) for ranks 2-6, a flat Range with index decomposition
// beyond.
template <class V, class F, class FlatF>
void for_each_index(const MI355X& exec, const char* label, const V& v, const F& f, const FlatF& flat) {
  constexpr unsigned R = V::rank;
  if constexpr (R == 1) {
    parallel_for(label, RangePolicy<MI355X, IndexType<int64_t>>(exec, 0, int64_t(v.extent(0))),
                 KOKKOS_LAMBDA(const int64_t i) { f(i); });
  } else if constexpr (R >= 2 && R <= 6) {
    constexpr Iterate it = std::is_same<typename V::array_layout, LayoutRight>::value ? Iterate::Right : Iterate::Left;
    using MP             = MDRangePolicy<MI355X, Rank<R, it, it>, IndexType<int64_t>>;
    typename MP::point_type lo{}, hi{};
    for (unsigned r = 0; r < R; ++r) {
      lo[r] = 0;
      hi[r] = static_cast<int64_t>(v.extent(r));
    }
    parallel_for(label, MP(exec, lo, hi), f);
  } else {
    parallel_for(label, RangePolicy<MI355X, IndexType<int64_t>>(exec, 0, int64_t(v.size())), flat);
  }
}

template <class Mem>
constexpr bool host_accessible() {
  return exec_can_access<Serial, Mem>::value;
}
template <class Mem>
constexpr bool device_accessible() {
  return exec_can_access<MI355X, Mem>::value;
}

template <class DV, class SV>
void check_shapes(const DV& dst, const SV& src) {
  static_assert(unsigned(DV::rank) == unsigned(SV::rank), "deep_copy: rank mismatch");
  for (unsigned r = 0; r < DV::rank; ++r)
    if (dst.extent(r) != src.extent(r))
      throw_runtime_exception("Deprecation Error: Kokkos::deep_copy extents of views don't match: " +
                              dst.label() + "(" + std::to_string(dst.extent(r)) + ") " + src.label() + "(" +
                              std::to_string(src.extent(r)) + ")");
}
}  // namespace Impl

namespace Impl {
// The same elements as v, as an unmanaged View in memory space Mem with v's
// extents and strides (a subview's strides are not implied by its extents).
template <class Mem, class V>
KOKKOS_INLINE_FUNCTION auto rewrap_unmanaged(const V& v) {
  using W = View<typename V::data_type, typename V::array_layout, Mem, MemoryTraits<Unmanaged>>;
  size_t ext[8], str[8];
  for (unsigned r = 0; r < 8; ++r) {
    ext[r] = v.extent(r);
    str[r] = r < V::rank ? v.stride(r) : 1;
  }
  return W(SubviewCtor{}, v.data(), ext, str, nullptr);
}

// ViewFill (reference core/src/Kokkos_CopyViews.hpp:58-260): one pass over
// the span when it is the index space, else over the index space.
template <class V>
void host_fill(const V& dst, const typename V::const_value_type& value) {
  if (dst.span_is_contiguous()) {
    auto* p = dst.data();
    for (size_t i = 0; i < dst.span(); ++i) p[i] = value;
  } else {
    auto h   = rewrap_unmanaged<HostSpace>(dst);
    using HV = decltype(h);
    IndexFill<HV> f{h, value};
    for (size_t i = 0; i < dst.size(); ++i) {
      size_t idx[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      size_t r      = i;
      for (int d = int(V::rank) - 1; d >= 0; --d) {
        idx[d] = r % dst.extent(d);
        r /= dst.extent(d);
      }
      if constexpr (V::rank == 0) f();
      else if constexpr (V::rank == 1) f(idx[0]);
      else if constexpr (V::rank == 2) f(idx[0], idx[1]);
      else if constexpr (V::rank == 3) f(idx[0], idx[1], idx[2]);
      else if constexpr (V::rank == 4) f(idx[0], idx[1], idx[2], idx[3]);
      else if constexpr (V::rank == 5) f(idx[0], idx[1], idx[2], idx[3], idx[4]);
      else if constexpr (V::rank == 6) f(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5]);
      else if constexpr (V::rank == 7) f(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5], idx[6]);
      else f(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5], idx[6], idx[7]);
    }
  }
}
template <class V>
void device_fill(const MI355X& exec, const V& dst, const typename V::const_value_type& value) {
  if (dst.span_is_contiguous()) {
    FillFunctor<V> f{dst.data(), value};
    parallel_for("Kokkos::ViewFill", RangePolicy<MI355X, IndexType<int64_t>>(exec, 0, int64_t(dst.span())), f);
    return;
  }
  auto u   = rewrap_unmanaged<MI355XSpace>(dst);
  using UV = decltype(u);
  IndexFill<UV> f{u, value};
  for_each_index(exec, "Kokkos::ViewFill", u, f, [=] KOKKOS_FUNCTION(const int64_t i) {
    size_t idx[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int64_t r     = i;
    for (int d = int(UV::rank) - 1; d >= 0; --d) {
      idx[d] = static_cast<size_t>(r % static_cast<int64_t>(u.extent(d)));
      r /= static_cast<int64_t>(u.extent(d));
    }
    if constexpr (UV::rank == 7) f(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5], idx[6]);
    else if constexpr (UV::rank == 8) f(idx[0], idx[1], idx[2], idx[3], idx[4], idx[5], idx[6], idx[7]);
  });
}
// ViewCopy between device-accessible Views (reference
// core/src/Kokkos_CopyViews.hpp:262-420): same layout and both spans
// contiguous -> one contiguous copy (8-byte words when sizes and alignment
// allow); LayoutLeft <-> LayoutRight -> the LDS-tiled transpose; otherwise
// an index-space copy in dst's layout order.
template <class DV, class SV>
void device_copy(const MI355X& exec, const DV& dst, const SV& src) {
  using T                = typename DV::non_const_value_type;
  const bool same_layout = std::is_same<typename DV::array_layout, typename SV::array_layout>::value || DV::rank <= 1;
  if (same_layout && dst.span_is_contiguous() && src.span_is_contiguous()) {
    const size_t bytes = dst.span() * sizeof(T);
    if (bytes % 8 == 0 && reinterpret_cast<uintptr_t>(dst.data()) % 8 == 0 &&
        reinterpret_cast<uintptr_t>(src.data()) % 8 == 0) {
      parallel_for("Kokkos::ViewCopy", RangePolicy<MI355X, IndexType<int64_t>>(exec, 0, int64_t(bytes / 8)),
                   CopyElems<uint64_t>{reinterpret_cast<const uint64_t*>(src.data()),
                                       reinterpret_cast<uint64_t*>(dst.data())});
    } else {
      parallel_for("Kokkos::ViewCopy", RangePolicy<MI355X, IndexType<int64_t>>(exec, 0, int64_t(dst.span())),
                   CopyElems<T>{src.data(), dst.data()});
    }
    return;
  }
  if (layout_transpose(exec, dst, src)) return;
  auto d   = rewrap_unmanaged<MI355XSpace>(dst);
  auto s   = rewrap_unmanaged<MI355XSpace>(typename SV::const_type(src));
  using UD = decltype(d);
  using US = decltype(s);
  IndexCopy<UD, US> f{d, s};
  ElementCopy<UD, US> flat{d, s};
  for_each_index(exec, "Kokkos::ViewCopy", d, f, flat);
}
}  // namespace Impl

// View <- scalar
template <class D, class... P>
inline void deep_copy(const View<D, P...>& dst, const typename View<D, P...>::const_value_type& value) {
  using V   = View<D, P...>;
  using Mem = typename V::memory_space;
  static_assert(!std::is_const<typename V::value_type>::value, "deep_copy into a const View");
  if (dst.span() == 0) return;
  Kokkos::fence("Kokkos::deep_copy: scalar copy, pre view equality check");
  if constexpr (Impl::host_accessible<Mem>()) {
    Impl::host_fill(dst, value);
  } else {
    Impl::device_fill(MI355X(), dst, value);
  }
  Kokkos::fence("Kokkos::deep_copy: scalar copy, post copy fence");
}
template <class E, class D, class... P,
          class = std::enable_if_t<is_execution_space<E>::value>>
inline void deep_copy(const E& exec, const View<D, P...>& dst,
                      const typename View<D, P...>::const_value_type& value) {
  using V   = View<D, P...>;
  using Mem = typename V::memory_space;
  if (dst.span() == 0) return;
  if constexpr (Impl::host_accessible<Mem>()) {
    exec.fence();
    Impl::host_fill(dst, value);
  } else if constexpr (std::is_same<E, MI355X>::value) {
    Impl::device_fill(exec, dst, value);
  } else {
    exec.fence();
    Impl::device_fill(MI355X(), dst, value);
    Kokkos::fence("Kokkos::deep_copy: fill on another space's instance");
  }
}

// scalar <- rank-0 View
template <class T, class S, class... P>
inline std::enable_if_t<!is_view<T>::value> deep_copy(T& dst, const View<S, P...>& src) {
  static_assert(View<S, P...>::rank == 0, "deep_copy(scalar, View) needs a rank-0 View");
  Kokkos::fence("Kokkos::deep_copy: copy into scalar, pre copy fence");
  KKMX_SAFE_CALL(mx_memcpy(&dst, src.data(), sizeof(T)));
}
// scalar <- rank-0 View, ordered on exec's stream; the value is valid after
// exec.fence().
template <class E, class T, class S, class... P,
          class = std::enable_if_t<is_execution_space<E>::value && !is_view<T>::value>>
inline void deep_copy(const E& exec, T& dst, const View<S, P...>& src) {
  static_assert(View<S, P...>::rank == 0, "deep_copy(exec, scalar, View) needs a rank-0 View");
  if constexpr (std::is_same<E, MI355X>::value) {
    KKMX_SAFE_CALL(mx_memcpy_async(&dst, src.data(), sizeof(T), exec.stream()));
  } else {
    exec.fence();
    KKMX_SAFE_CALL(mx_memcpy(&dst, src.data(), sizeof(T)));
  }
}
// rank-0 View <- scalar handled by the scalar fill overload above.

// View <- View
template <class D1, class... P1, class D2, class... P2>
inline void deep_copy(const View<D1, P1...>& dst, const View<D2, P2...>& src) {
  using DV = View<D1, P1...>;
  using SV = View<D2, P2...>;
  static_assert(std::is_same<typename DV::non_const_value_type, typename SV::non_const_value_type>::value,
                "deep_copy requires matching value types");
  if (dst.data() == nullptr && src.data() == nullptr) return;
  Impl::check_shapes(dst, src);
  if (dst.data() == src.data() && dst.span() == src.span()) {
    Kokkos::fence("Kokkos::deep_copy: copy between contiguous views, fence due to same spans");
    return;
  }
  Kokkos::fence("Kokkos::deep_copy: copy between views, pre view equality check");
  const bool same_layout = std::is_same<typename DV::array_layout, typename SV::array_layout>::value || DV::rank <= 1;
  constexpr bool both_device = Impl::device_accessible<typename DV::memory_space>() &&
                               Impl::device_accessible<typename SV::memory_space>();
  if constexpr (both_device) {
    Impl::device_copy(MI355X(), dst, src);
  } else if (same_layout && dst.span_is_contiguous() && src.span_is_contiguous()) {
    KKMX_SAFE_CALL(mx_memcpy(dst.data(), src.data(), dst.span() * sizeof(typename DV::value_type)));
  } else if constexpr (Impl::host_accessible<typename DV::memory_space>() &&
                       Impl::host_accessible<typename SV::memory_space>()) {
    Impl::ElementCopy<DV, SV> f{dst, src};
    for (int64_t i = 0; i < int64_t(dst.size()); ++i) f(i);
  } else {
    // Across spaces with different layouts or a non-contiguous operand:
    // rearrange on whichever side can index both Views, with one contiguous
    // transfer of a same-layout staging buffer in between.
    using T = typename DV::non_const_value_type;
    if constexpr (Impl::host_accessible<typename DV::memory_space>()) {
      // device -> host: reorder on the device into dst's layout, then copy
      View<typename DV::traits::non_const_data_type, typename DV::array_layout, MI355XSpace> stage(
          view_alloc(WithoutInitializing, std::string("deep_copy_stage")), Impl::compact_layout(dst));
      Impl::device_copy(MI355X(), stage, src);
      MI355X().fence("Kokkos::deep_copy: staged device copy");
      if (dst.span_is_contiguous()) {
        KKMX_SAFE_CALL(mx_memcpy(dst.data(), stage.data(), dst.size() * sizeof(T)));
      } else {
        auto hs = create_mirror(stage);
        KKMX_SAFE_CALL(mx_memcpy(hs.data(), stage.data(), dst.size() * sizeof(T)));
        Impl::ElementCopy<DV, decltype(hs)> f{dst, hs};
        for (int64_t i = 0; i < int64_t(dst.size()); ++i) f(i);
      }
    } else {
      // host -> device: a contiguous host copy in src's layout, one transfer,
      // then reorder on the device
      typename SV::HostMirror hs(view_alloc(WithoutInitializing, std::string("deep_copy_stage")), Impl::compact_layout(src));
      Impl::ElementCopy<typename SV::HostMirror, SV> f{hs, src};
      for (int64_t i = 0; i < int64_t(src.size()); ++i) f(i);
      View<typename SV::traits::non_const_data_type, typename SV::array_layout, MI355XSpace> stage(
          view_alloc(WithoutInitializing, std::string("deep_copy_stage")), Impl::compact_layout(src));
      KKMX_SAFE_CALL(mx_memcpy(stage.data(), hs.data(), src.size() * sizeof(T)));
      Impl::device_copy(MI355X(), dst, stage);
      MI355X().fence("Kokkos::deep_copy: staged device copy");
    }
  }
  Kokkos::fence("Kokkos::deep_copy: copy between views, post deep copy fence");
}

template <class E, class D1, class... P1, class D2, class... P2,
          class = std::enable_if_t<is_execution_space<E>::value>>
inline void deep_copy(const E& exec, const View<D1, P1...>& dst, const View<D2, P2...>& src) {
  using DV = View<D1, P1...>;
  using SV = View<D2, P2...>;
  Impl::check_shapes(dst, src);
  const bool same_layout = std::is_same<typename DV::array_layout, typename SV::array_layout>::value || DV::rank <= 1;
  if constexpr (std::is_same<E, MI355X>::value && Impl::device_accessible<typename DV::memory_space>() &&
                Impl::device_accessible<typename SV::memory_space>()) {
    // ordered on exec's stream, no fence
    if (dst.data() != src.data() || dst.span() != src.span()) Impl::device_copy(exec, dst, src);
    return;
  }
  if (!(same_layout && dst.span_is_contiguous() && src.span_is_contiguous()))
    return deep_copy(dst, src);
  if constexpr (std::is_same<E, MI355X>::value) {
    KKMX_SAFE_CALL(mx_memcpy_async(dst.data(), src.data(), dst.span() * sizeof(typename DV::value_type),
                                   exec.stream()));
  } else {
    exec.fence();
    std::memcpy(static_cast<void*>(dst.data()), src.data(), dst.span() * sizeof(typename DV::value_type));
  }
}

// ------------------------------------------------------------------ mirrors
template <class D, class... P>
inline typename View<D, P...>::HostMirror create_mirror(const View<D, P...>& v) {
  using M = typename View<D, P...>::HostMirror;
  return M(view_alloc(v.label() + "_mirror"), v.layout());
}
template <class D, class... P>
inline typename View<D, P...>::HostMirror create_mirror(Impl::WithoutInitializing_t, const View<D, P...>& v) {
  using M = typename View<D, P...>::HostMirror;
  return M(view_alloc(WithoutInitializing, v.label() + "_mirror"), v.layout());
}
template <class Space, class D, class... P,
          class = std::enable_if_t<is_memory_space<Space>::value || is_execution_space<Space>::value>>
inline auto create_mirror(const Space&, const View<D, P...>& v) {
  using Mem = typename Space::memory_space;
  using M   = View<typename View<D, P...>::traits::non_const_data_type, typename View<D, P...>::array_layout, Mem>;
  return M(view_alloc(v.label() + "_mirror"), v.layout());
}

template <class D, class... P>
inline auto create_mirror_view(const View<D, P...>& v) {
  using V = View<D, P...>;
  if constexpr (Impl::host_accessible<typename V::memory_space>() &&
                std::is_same<typename V::HostMirror::memory_space, typename V::memory_space>::value &&
                std::is_same<typename V::value_type, typename V::non_const_value_type>::value) {
    return typename V::HostMirror(v);
  } else {
    return create_mirror(v);
  }
}
template <class D, class... P>
inline auto create_mirror_view(Impl::WithoutInitializing_t, const View<D, P...>& v) {
  using V = View<D, P...>;
  if constexpr (Impl::host_accessible<typename V::memory_space>() &&
                std::is_same<typename V::HostMirror::memory_space, typename V::memory_space>::value &&
                std::is_same<typename V::value_type, typename V::non_const_value_type>::value) {
    return typename V::HostMirror(v);
  } else {
    return create_mirror(WithoutInitializing, v);
  }
}
template <class Space, class D, class... P,
          class = std::enable_if_t<is_memory_space<Space>::value || is_execution_space<Space>::value>>
inline auto create_mirror_view(const Space& s, const View<D, P...>& v) {
  using Mem = typename Space::memory_space;
  using V   = View<D, P...>;
  using M   = View<typename V::traits::non_const_data_type, typename V::array_layout, Mem>;
  if constexpr (std::is_same<typename V::memory_space, Mem>::value &&
                std::is_same<typename V::value_type, typename V::non_const_value_type>::value) {
    return M(v);
  } else {
    return create_mirror(s, v);
  }
}
template <class Space, class D, class... P,
          class = std::enable_if_t<is_memory_space<Space>::value || is_execution_space<Space>::value>>
inline auto create_mirror_view_and_copy(const Space& s, const View<D, P...>& v) {
  using Mem = typename Space::memory_space;
  using V   = View<D, P...>;
  using M   = View<typename V::traits::non_const_data_type, typename V::array_layout, Mem>;
  if constexpr (std::is_same<typename V::memory_space, Mem>::value &&
                std::is_same<typename V::value_type, typename V::non_const_value_type>::value) {
    Kokkos::fence("Kokkos::create_mirror_view_and_copy: fence before returning src view");
    return M(v);
  } else {
    M m(view_alloc(WithoutInitializing, v.label() + "_mirror"), v.layout());
    deep_copy(m, v);
    return m;
  }
}

// ------------------------------------------------------------------ resize / realloc
template <class D, class... P>
inline void realloc(View<D, P...>& v, size_t n0 = 0, size_t n1 = 0, size_t n2 = 0, size_t n3 = 0) {
  using V     = View<D, P...>;
  std::string l = v.label();
  v           = V();
  v           = V(l, n0, n1, n2, n3);
}
// Keeps every element whose indices fit both the old and the new extents,
// element by element (core/src/Kokkos_CopyViews.hpp:690-800, ViewRemap, and
// :2512-2650, impl_resize): the common box of the two Views, seen through
// strided windows, is deep-copied.
template <class D, class... P>
inline void resize(View<D, P...>& v, size_t n0 = 0, size_t n1 = 0, size_t n2 = 0, size_t n3 = 0) {
  using V = View<D, P...>;
  V nv(v.label(), n0, n1, n2, n3);
  if (v.data() && nv.data()) {
    LayoutStride from, to;
    for (unsigned r = 0; r < V::rank; ++r) {
      const size_t common = v.extent(r) < nv.extent(r) ? v.extent(r) : nv.extent(r);
      from.dimension[r] = to.dimension[r] = common;
      from.stride[r]    = v.stride(r);
      to.stride[r]      = nv.stride(r);
    }
    using W = View<typename V::data_type, LayoutStride, typename V::device_type, MemoryTraits<Unmanaged>>;
    deep_copy(W(nv.data(), to), W(v.data(), from));
  }
  v = nv;
}

}  // namespace Kokkos

#endif
