// Device LSD radix sort for MI355X (gfx950): 8-bit digits over the unsigned
// image of 4- and 8-byte arithmetic keys, alone or with a 4- or 8-byte
// payload word per key.
//
// A pass is two or three launches.  k_radix_count counts the digit in every
// segment (the consecutive tiles of one block), k_radix_offsets turns the
// counts into each segment's first output positions, and k_radix_scatter
// ranks a tile's keys in LDS and writes them out as one contiguous run per
// digit, stably; up to kRadixDirect segments it adds up the counts by itself.
// The first count also folds the AND and OR of all keys: digits where the two
// agree are the same in every key and need no pass, which the device decides by
// itself.  8-byte keys are sorted by their five highest digits that vary where a
// sample shows those to tell them apart (k_radix_sample), and neighbours that
// share them are put right on the way back (k_radix_finish).  A sort is a fixed
// sequence of launches and one wait, two for 8-byte keys that are not trimmed,
// and more where many keys share those digits after all (radix_sort_long_runs).
// Few keys are sorted in LDS: those of one block by a single launch
// (k_radix_small), those of several blocks' runs by one more that places every
// key among the other runs (k_radix_merge).
//
// Reading the keys twice a pass costs less than learning the positions in one
// sweep: a decoupled look-back over tiles took 0.42 ms of a 1.0 ms pass over
// 2^28 32-bit keys (its 256 status words per 8192-key tile are walked across
// the tiles in flight), the count takes 0.2 ms.
//
// Floating-point keys sort as operator< orders them: -0.0 and +0.0 compare
// equal and keep their input order; NaNs go below -inf (sign bit set) or
// above +inf.
#ifndef KKMX_RADIXSORT_HPP
#define KKMX_RADIXSORT_HPP

#include <Kokkos_Core.hpp>

#include <mutex>

namespace Kokkos {
namespace Impl {

template <class T>
struct RadixKey {
  using U = std::conditional_t<sizeof(T) == 4, uint32_t, uint64_t>;
  static constexpr U top      = U(1) << (8 * sizeof(T) - 1);
  static constexpr int passes = int(sizeof(T));
  KOKKOS_FORCEINLINE_FUNCTION static U encode(U u) {
    if constexpr (std::is_floating_point<T>::value) return (u & top) ? ~u : (u | top);
    else if constexpr (std::is_signed<T>::value) return u ^ top;
    else return u;
  }
  KOKKOS_FORCEINLINE_FUNCTION static U decode_if(U u, bool yes) { return yes ? decode(u) : u; }
  KOKKOS_FORCEINLINE_FUNCTION static U decode(U u) {
    if constexpr (std::is_floating_point<T>::value) return (u & top) ? (u ^ top) : ~u;
    else if constexpr (std::is_signed<T>::value) return u ^ top;
    else return u;
  }
  // -0.0 (encoded ~top) takes the digits of +0.0 (encoded top), so the two
  // compare equal and keep their input order; the key itself keeps its bits.
  KOKKOS_FORCEINLINE_FUNCTION static U canon(U u) {
    if constexpr (std::is_floating_point<T>::value) return u == U(~top) ? top : u;
    else return u;
  }
  KOKKOS_FORCEINLINE_FUNCTION static unsigned digit(U u, int shift) { return unsigned(canon(u) >> shift) & 255u; }
};

// No payload: keys alone are sorted.
struct NoPayload {};

// AND and OR of the canonical keys of a sort.  Two of them alternate between
// calls: the first count of a call folds into its own and clears the other.
struct RadixSummary {
  unsigned long long all, any;
};
struct RadixControl {
  RadixSummary summary[2];
  uint32_t totals[256];
  uint32_t trim;  // 8-byte keys: only the kRadixTrim highest digits that vary are sorted
};

// Random 8-byte keys differ in their highest five or so digits: sorting by
// those leaves a few neighbours that share them out of order, which
// k_radix_finish puts right.  The digits are trimmed where at least two more
// would be sorted and a sample of the keys shows no crowding.
constexpr int kRadixTrim = 5;

// What a pass does, from the digits that vary.  Passes run on alternate
// buffers and the result belongs in the caller's, so their number is even: an
// odd count takes in one digit that need not move, and a permutation of keys
// that are in order already (Iota) is written by two.  Trimmed passes end in
// the second buffers, still encoded, and k_radix_finish takes them back.
struct RadixPlan {
  bool run, from_second, first, last;
  int digit;
};
template <class T>
__device__ __forceinline__ unsigned radix_varying(const RadixSummary& s) {
  const unsigned long long vary = s.all ^ s.any;
  unsigned digits               = 0;
#pragma unroll
  for (int q = 0; q < RadixKey<T>::passes; ++q) digits |= ((vary >> (8 * q)) & 255u) ? 1u << q : 0u;
  return digits;
}
// The digits that passes sort by.
template <class T, bool Iota>
__device__ __forceinline__ unsigned radix_digits(const RadixSummary& s, bool trim) {
  unsigned runs = radix_varying<T>(s);
  if (trim) {
    while (__builtin_popcount(runs) > kRadixTrim) runs &= runs - 1;
    return runs;
  }
  const int want = (Iota && runs == 0) ? 2 : (__builtin_popcount(runs) + 1) & ~1;
#pragma unroll
  for (int q = 0; q < RadixKey<T>::passes; ++q)
    if (__builtin_popcount(runs) < want) runs |= 1u << q;
  return runs;
}
// Pass p of a sort: digit p of 4-byte keys, the p-th digit to be sorted of
// 8-byte keys.  p < 0 is a single pass of its own, outside a sort: from the
// first buffers to the second, keys as they are.
template <class T, bool Iota>
__device__ __forceinline__ RadixPlan radix_plan(const RadixControl* ctl, int turn, int p) {
  if (p < 0) return {true, false, false, false, 0};
  const bool trim     = sizeof(T) == 8 && ctl->trim != 0;
  const unsigned runs = radix_digits<T, Iota>(ctl->summary[turn], trim);
  int digit           = p;
  if constexpr (sizeof(T) == 8) {
    unsigned left = runs;
    for (int q = 0; q < p; ++q) left &= left - 1;
    if (left == 0) return {false, false, false, false, 0};
    digit = __builtin_ctz(left);
  }
  const unsigned below = runs & ((1u << digit) - 1);
  return {((runs >> digit) & 1u) != 0, (__builtin_popcount(below) & 1) != 0, below == 0,
          !trim && (runs >> digit) == 1u, digit};
}

// Counts of one digit per segment, counts[segment * 256 + d].  It reads at
// the rate of a copy's read half as long as the LDS atomics keep up, one per
// key: a bin has 16 counters, adjacent in LDS, one for every 16th lane, so
// lanes of different groups never meet in a bank, and keys that share a digit
// (the exponents of floating-point keys, small ranges) only within a group.
constexpr int kRadixCountLanes = 512;
template <class T, bool Iota>
__global__ __launch_bounds__(kRadixCountLanes) void k_radix_count(const int p, const int pass_shift,
                                                                  const int64_t n, const int64_t segment,
                                                                  const typename RadixKey<T>::U* k0,
                                                                  const typename RadixKey<T>::U* k1, RadixControl* ctl,
                                                                  const int turn, const bool fold, uint32_t* counts) {
  using R             = RadixKey<T>;
  using U             = typename R::U;
  constexpr int C     = 16;
  constexpr int Items = 64 / sizeof(U);
  __shared__ uint32_t h[256 * C];
  __shared__ unsigned long long s_all, s_any;
  const int t = threadIdx.x, l = t & 63;
  RadixPlan plan{true, false, true, false, 0};
  if (!fold) plan = radix_plan<T, Iota>(ctl, turn, p);
  if (!plan.run) return;
  if (!fold && p == 0 && plan.digit == 0) return;  // counted by the fold
  const int shift = p < 0 ? pass_shift : 8 * plan.digit;
  const U* in = plan.from_second ? k1 : k0;
  for (int k = t; k < 256 * C; k += kRadixCountLanes) h[k] = 0;
  if (t == 0) s_all = ~0ull, s_any = 0ull;
  __syncthreads();
  const int c = l & (C - 1);
  U all = ~U(0), any = U(0);
  const int64_t first = int64_t(blockIdx.x) * segment;
  const int64_t last  = first + segment < n ? first + segment : n;
  constexpr int Step  = kRadixCountLanes * Items;
  for (int64_t b = first; b < last; b += Step) {
    const U* from  = in + b;
    const int left = last - b < Step ? int(last - b) : Step;
    U u[Items];
    if (left == Step) {
#pragma unroll
      for (int r = 0; r < Items; ++r) u[r] = from[r * kRadixCountLanes + t];
    } else {
#pragma unroll
      for (int r = 0; r < Items; ++r) u[r] = r * kRadixCountLanes + t < left ? from[r * kRadixCountLanes + t] : U(0);
    }
#pragma unroll
    for (int r = 0; r < Items; ++r) {
      if (left == Step || r * kRadixCountLanes + t < left) {
        const U k = R::canon(plan.first ? R::encode(u[r]) : u[r]);
        atomicAdd(&h[(unsigned(k >> shift) & 255u) * C + c], 1u);
        if (fold) all &= k, any |= k;
      }
    }
  }
  if (fold) {
    atomicAnd(&s_all, (unsigned long long)all);
    atomicOr(&s_any, (unsigned long long)any);
  }
  __syncthreads();
  if (t < 256) {
    uint32_t s = 0;
#pragma unroll
    for (int q = 0; q < C; ++q) s += h[t * C + ((q + l) & (C - 1))];
    counts[int64_t(blockIdx.x) * 256 + t] = s;
  }
  if (fold && t == 0) {
    atomicAnd(&ctl->summary[turn].all, s_all);
    atomicOr(&ctl->summary[turn].any, s_any);
    if (blockIdx.x == 0) ctl->summary[turn ^ 1] = {~0ull, 0ull};
  }
}

// counts[segment * 256 + d] becomes the number of keys with digit d in the
// segments before; totals[d] their number in all.  One wavefront takes 4
// digits (16 bytes a segment and lane row) through the segments, 64 of them
// per round.
constexpr int kRadixOffsetLanes = 1024;
template <class T, bool Iota>
__global__ __launch_bounds__(kRadixOffsetLanes) void k_radix_offsets(const int p, RadixControl* ctl, const int turn,
                                                                     uint32_t* counts, const int segments) {
  if (!radix_plan<T, Iota>(ctl, turn, p).run) return;
  __shared__ uint32_t s_sum[16][4];
  const int t = threadIdx.x, w = t >> 6, l = t & 63;
  uint4* col      = reinterpret_cast<uint4*>(counts) + blockIdx.x;  // 4 digits of segment 0
  const auto plus = [](uint32_t& a, const uint32_t& x) { a += x; };
  uint4 carry{0, 0, 0, 0};
  for (int b = 0; b < segments; b += kRadixOffsetLanes) {
    const int i = b + t;
    const uint4 x = i < segments ? col[int64_t(i) * 64] : uint4{0, 0, 0, 0};
    uint4 inc;
    inc.x = wave::inclusive_scan(x.x, 0u, plus);
    inc.y = wave::inclusive_scan(x.y, 0u, plus);
    inc.z = wave::inclusive_scan(x.z, 0u, plus);
    inc.w = wave::inclusive_scan(x.w, 0u, plus);
    if (l == 63) s_sum[w][0] = inc.x, s_sum[w][1] = inc.y, s_sum[w][2] = inc.z, s_sum[w][3] = inc.w;
    __syncthreads();
    uint4 before = carry;
    for (int q = 0; q < 16; ++q) {
      if (q < w) before.x += s_sum[q][0], before.y += s_sum[q][1], before.z += s_sum[q][2], before.w += s_sum[q][3];
      carry.x += s_sum[q][0], carry.y += s_sum[q][1], carry.z += s_sum[q][2], carry.w += s_sum[q][3];
    }
    if (i < segments)
      col[int64_t(i) * 64] = uint4{before.x + inc.x - x.x, before.y + inc.y - x.y, before.z + inc.z - x.z,
                                   before.w + inc.w - x.w};
    __syncthreads();
  }
  if (t == 0) reinterpret_cast<uint4*>(ctl->totals)[blockIdx.x] = carry;
}

// Rank of every key among its wavefront's keys of the same digit, in order of
// position.  Eight ballots per 64 keys give each lane the lanes that share
// its digit; the lowest of them adds their number to the wavefront's LDS
// counter and every lane reads the counter back.  A wavefront's LDS
// operations execute in order, so the rounds' adds and reads are all in
// flight together and no round waits for the one before it.
template <class R, int Items>
__device__ __forceinline__ void radix_rank(const typename R::U (&u)[Items], uint32_t (&rank)[Items], int shift,
                                           uint32_t* cnt, int rounds = Items) {
  uint32_t seen[Items];
#pragma unroll
  for (int r = 0; r < Items; ++r) {
    if (r >= rounds) break;
    const unsigned d = R::digit(u[r], shift);
    uint32_t lo = ~0u, hi = ~0u;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      int32_t xb = __builtin_amdgcn_sbfe(int32_t(d), b, 1);  // 0 or all ones
      asm("" : "+v"(xb));  // one extract serves the compare and the select
      const uint64_t m = __builtin_amdgcn_ballot_w64(xb != 0);
      // lo & ~(m ^ xb): lanes whose bit b is this lane's
      lo = __builtin_amdgcn_bitop3_b32(lo, uint32_t(m), uint32_t(xb), 0x90);
      hi = __builtin_amdgcn_bitop3_b32(hi, uint32_t(m >> 32), uint32_t(xb), 0x90);
    }
    const uint32_t below = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
    const uint32_t total = uint32_t(__popc(lo)) + uint32_t(__popc(hi));
    if (below == 0) __hip_atomic_fetch_add(&cnt[d], total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    seen[r] = __hip_atomic_load(&cnt[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    rank[r] = below - total;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
#pragma unroll
  for (int r = 0; r < Items; ++r)
    if (r < rounds) rank[r] += seen[r];
}

// Exclusive prefix over the 256 threads of wavefronts 0-3 (other wavefronts
// only take part in the barrier).
template <int NW>
__device__ __forceinline__ uint32_t radix_prefix256(uint32_t x, uint32_t* s_wave) {
  const auto plus    = [](uint32_t& a, const uint32_t& y) { a += y; };
  const int w        = threadIdx.x >> 6;
  const uint32_t inc = wave::inclusive_scan(x, 0u, plus);
  if (w < 4 && wave::lane() == 63) s_wave[w] = inc;
  __syncthreads();
  uint32_t before = 0;
#pragma unroll
  for (int q = 0; q < 3; ++q) before += (q < w) ? s_wave[q] : 0u;
  return before + inc - x;
}

// Up to this many segments the scatter adds up the counts before its own by
// itself, which is shorter than another launch.
constexpr int kRadixDirect = 48;

// One digit, one segment per block, tile after tile of Lanes x Items keys;
// wavefront w holds a run of 64 * Items of them.  Thread d < 256 carries digit
// d's next output position from tile to tile, and the next tile's keys are
// loaded before this one is written out.  `summed` says that k_radix_offsets has
// been over the counts; else they are the segments' own, added up here.
template <class T, class PT, bool Iota, int Lanes, int Items>
__global__ __launch_bounds__(Lanes, 4) void k_radix_scatter(
    const int p, const int pass_shift, const int64_t n, const int64_t segment, const typename RadixKey<T>::U* k0,
    typename RadixKey<T>::U* k1, const PT* p0, PT* p1, const RadixControl* ctl, const int turn, const uint32_t* counts,
    const bool summed) {
  using R              = RadixKey<T>;
  using U              = typename R::U;
  constexpr bool Pairs = !std::is_same<PT, NoPayload>::value;
  constexpr int NW     = Lanes / 64;
  constexpr int Tile   = Lanes * Items;
  using Wide           = std::conditional_t<(Pairs && sizeof(PT) > sizeof(U)), uint64_t, U>;
  __shared__ Wide s_tile[Tile];  // the tile's keys, then its payload, in digit order
  __shared__ uint32_t wcnt[NW][256];
  __shared__ uint32_t gshift[256];  // output position of tile slot j of digit d: gshift[d] + j
  __shared__ uint32_t s_wave[4];
  const RadixPlan plan = radix_plan<T, Iota>(ctl, turn, p);
  if (!plan.run) return;
  const int shift = p < 0 ? pass_shift : 8 * plan.digit;
  // k0 and p0 are only written by passes that read the second buffers
  const U* in    = plan.from_second ? k1 : k0;
  U* out         = plan.from_second ? const_cast<U*>(k0) : k1;
  const PT* in_p = plan.from_second ? p1 : p0;
  PT* out_p      = plan.from_second ? const_cast<PT*>(p0) : p1;
  U* key_tile    = reinterpret_cast<U*>(s_tile);
  PT* pay_tile   = reinterpret_cast<PT*>(s_tile);
  const int t = threadIdx.x, l = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  U u[Items];
  PT v[Pairs ? Items : 1];
  // Keys of the tile at `tfirst`; past the end of the last one they are all
  // ones, which keeps them behind every key of the tile in every pass.
  const auto load = [&](int64_t tfirst) {
    const int64_t wfirst = tfirst + w * (64 * Items);
    const U* from        = in + wfirst;
    const int left       = n - wfirst < 64 * Items ? int(n - wfirst) : 64 * Items;
    if (left == 64 * Items) {
#pragma unroll
      for (int r = 0; r < Items; ++r) u[r] = from[r * 64 + l];
    } else {
#pragma unroll
      for (int r = 0; r < Items; ++r) u[r] = r * 64 + l < left ? from[r * 64 + l] : R::decode_if(~U(0), plan.first);
    }
    if constexpr (Pairs) {
      if (!(Iota && plan.first)) {
        const PT* from_p = in_p + wfirst;
#pragma unroll
        for (int r = 0; r < Items; ++r) v[r] = r * 64 + l < left ? from_p[r * 64 + l] : PT(0);
      }
    }
  };
  const int64_t begin = int64_t(blockIdx.x) * segment;
  const int64_t end   = begin + segment < n ? begin + segment : n;
  load(begin);
  for (int k = t; k < NW * 256; k += Lanes) (&wcnt[0][0])[k] = 0;
  uint32_t next_pos = 0;  // of digit t
  {
    uint32_t total = 0;
    if (t < 256) {
      if (!summed) {
#pragma unroll 16
        for (int q = 0; q < int(gridDim.x); ++q) {
          const uint32_t x = counts[q * 256 + t];
          total += x;
          next_pos += q < int(blockIdx.x) ? x : 0u;
        }
      } else {
        total    = ctl->totals[t];
        next_pos = counts[int64_t(blockIdx.x) * 256 + t];
      }
    }
    next_pos += radix_prefix256<NW>(total, s_wave);
    __syncthreads();
  }
  for (int64_t tfirst = begin; tfirst < end; tfirst += Tile) {
    const int have = end - tfirst < Tile ? int(end - tfirst) : Tile;
    uint32_t slot[Items];
    if constexpr (Iota) {
      if (plan.first) {
#pragma unroll
        for (int r = 0; r < Items; ++r) v[r] = PT(tfirst + w * (64 * Items) + r * 64 + l);
      }
    }
    if (plan.first) {
#pragma unroll
      for (int r = 0; r < Items; ++r) u[r] = R::encode(u[r]);
    }
    radix_rank<R>(u, slot, shift, wcnt[w]);
    __syncthreads();  // the wavefronts' counts are complete
    uint32_t count = 0;
    if (t < 256) {
#pragma unroll
      for (int q = 0; q < NW; ++q) count += wcnt[q][t];
    }
    uint32_t at = radix_prefix256<NW>(count, s_wave);
    if (t < 256) {
      gshift[t] = next_pos - at;
      next_pos += count;
#pragma unroll 4
      for (int q = 0; q < NW; ++q) {
        const uint32_t c = wcnt[q][t];
        wcnt[q][t]       = at;
        at += c;
      }
    }
    __syncthreads();  // slot bases and output shifts visible
#pragma unroll
    for (int r = 0; r < Items; ++r) {
      slot[r] += wcnt[w][R::digit(u[r], shift)];
      key_tile[slot[r]] = u[r];
    }
    __syncthreads();  // tile in digit order
    const bool more = tfirst + Tile < end;
    for (int k = t; k < NW * 256; k += Lanes) (&wcnt[0][0])[k] = 0;
    if constexpr (!Pairs) {
      if (more) load(tfirst + Tile);
    }
    if constexpr (!Pairs) {
#pragma unroll 4
      for (int r = 0; r < Items; ++r) {
        const int j = r * Lanes + t;
        if (j < have) {
          U k                = key_tile[j];
          const uint32_t pos = gshift[R::digit(k, shift)] + uint32_t(j);
          if (plan.last) k = R::decode(k);
          out[pos] = k;
        }
      }
    } else {
      uint32_t to[Items];
#pragma unroll
      for (int r = 0; r < Items; ++r) {
        const int j = r * Lanes + t;
        if (j < have) {
          U k   = key_tile[j];
          to[r] = gshift[R::digit(k, shift)] + uint32_t(j);
          if (plan.last) k = R::decode(k);
          out[to[r]] = k;
        }
      }
      __syncthreads();  // the keys have left the tile
#pragma unroll
      for (int r = 0; r < Items; ++r) pay_tile[slot[r]] = v[r];
      __syncthreads();
      if (more) load(tfirst + Tile);
#pragma unroll
      for (int r = 0; r < Items; ++r) {
        const int j = r * Lanes + t;
        if (j < have) out_p[to[r]] = pay_tile[j];
      }
    }
    __syncthreads();  // the tile has left LDS, the counters are clear
  }
}

// Whether the digits of 8-byte keys are trimmed: 4096 keys, evenly spaced, go
// into an LDS hash table by their trimmed digits, and different keys that meet
// there are counted.  If all of n keys lie in runs of 64, which is more than
// k_radix_finish takes, 4096^2 / 2 * 64 / n meet: 8 at n = 2^26, more below.
// One block, bound by its loads' latency.
constexpr int kRadixSample = 4096;
template <class T>
__global__ __launch_bounds__(1024) void k_radix_sample(const typename RadixKey<T>::U* in, const int64_t n,
                                                       RadixControl* ctl, const int turn, const bool allow) {
  using R = RadixKey<T>;
  using U = typename R::U;
  __shared__ unsigned long long table[2 * kRadixSample];
  __shared__ unsigned met;
  const int t            = threadIdx.x;
  const unsigned digits  = radix_digits<T, false>(ctl->summary[turn], true);
  const bool worth       = allow && __builtin_popcount(radix_varying<T>(ctl->summary[turn])) >= kRadixTrim + 2;
  if (!worth) {
    if (t == 0) ctl->trim = 0;
    return;
  }
  const int low = 8 * __builtin_ctz(digits);
  for (int k = t; k < 2 * kRadixSample; k += 1024) table[k] = ~0ull;
  if (t == 0) met = 0;
  __syncthreads();
  const int64_t step = n / kRadixSample;
  for (int k = t; k < kRadixSample; k += 1024) {
    const unsigned long long key = R::canon(R::encode(in[k * step]));
    if (key == ~0ull) continue;
    unsigned at = unsigned(((key >> low) * 0x9E3779B97F4A7C15ull) >> 51);  // 13 bits
    for (int probe = 0; probe < 32; ++probe, at = (at + 1) & (2 * kRadixSample - 1)) {
      const unsigned long long was = atomicCAS(&table[at], ~0ull, key);
      if (was == ~0ull || was == key) break;
      if ((was >> low) == (key >> low)) {
        atomicAdd(&met, 1u);
        break;
      }
    }
  }
  __syncthreads();
  if (t == 0) ctl->trim = met <= 4 ? 1 : 0;
}

// Takes keys sorted by their trimmed digits from the second buffers to the
// caller's.  Neighbours that share those digits form a run; a key's place in
// its run is the number of keys before it there, by value, then by position.
// Most keys have no such neighbour, or a run already in order, which a
// wavefront sees from its own and the neighbouring wavefronts' ballots.  A run
// of 64 keys or more (every key of it sees that) is left as it is, and reported
// where it is out of order (status[0] 1, status[1] the lowest bit sorted by): the
// caller's keys are then still a stable order by the trimmed digits, and the keys
// of such runs are sorted by themselves (radix_sort_long_runs).  Status 2 reports
// digits left to sort where nothing was trimmed.
constexpr int kRadixRun         = 64;
constexpr int kRadixFinishLanes = 1024;
constexpr int kRadixFinishTile  = 4096;
// How far key j moves within its run.
template <class R, class U, class Tied>
__device__ __forceinline__ int radix_place_in_run(const U* s_key, const int j, const Tied& tied, bool& broken) {
  const U key = R::canon(s_key[j]);
  int lo = j, hi = j + 1;  // the run, as far as 64 keys to each side
  while (j - lo < kRadixRun - 1 && tied(lo)) --lo;
  while (hi - j < kRadixRun && tied(hi)) ++hi;
  if (tied(lo) || hi - j == kRadixRun || hi - lo >= kRadixRun) {
    for (int k = lo + 1; k < hi; ++k) broken = broken || R::canon(s_key[k]) < R::canon(s_key[k - 1]);
    return 0;
  }
  int before = 0;
  for (int k = lo; k < hi; ++k) {
    const U x = R::canon(s_key[k]);
    before += (x < key || (x == key && k < j)) ? 1 : 0;
  }
  return lo + before - j;
}

template <class T, class PT>
__global__ __launch_bounds__(kRadixFinishLanes) void k_radix_finish(const int64_t n, typename RadixKey<T>::U* k0,
                                                                    const typename RadixKey<T>::U* k1, PT* p0,
                                                                    const PT* p1, const RadixControl* ctl,
                                                                    const int turn, uint32_t* status) {
  using R              = RadixKey<T>;
  using U              = typename R::U;
  constexpr bool Pairs = !std::is_same<PT, NoPayload>::value;
  constexpr int NW     = kRadixFinishLanes / 64;
  constexpr int Items  = kRadixFinishTile / kRadixFinishLanes;
  const unsigned runs  = radix_digits<T, false>(ctl->summary[turn], ctl->trim != 0);
  const int t = threadIdx.x, w = t >> 6, l = t & 63;
  if (!ctl->trim) {
    if (blockIdx.x == 0 && t == 0 && __builtin_popcount(runs) > kRadixTrim) *status = 2;
    return;
  }
  const int low = 8 * __builtin_ctz(runs);
  // key base + x is s_key[x + kRadixRun + 1]; [0] is one before the halo
  __shared__ U s_key[kRadixFinishTile + 2 * kRadixRun + 1];
  // keys tied to the one before, and descents there, 64 keys a word, with a
  // word for each halo
  __shared__ uint64_t s_tied[kRadixFinishTile / 64 + 2], s_down[kRadixFinishTile / 64 + 2];
  bool broken = false;
  for (int64_t base = int64_t(blockIdx.x) * kRadixFinishTile; base < n; base += int64_t(gridDim.x) * kRadixFinishTile) {
    U raw[Items], halo = U(0);
    PT v[Pairs ? Items : 1];
#pragma unroll
    for (int r = 0; r < Items; ++r) {
      const int64_t i = base + r * kRadixFinishLanes + t;
      raw[r]          = i < n ? k1[i] : U(0);
      if constexpr (Pairs) {
        if (i < n) v[r] = p1[i];
      }
    }
    const int hj = t <= kRadixRun ? t : kRadixFinishTile + t;  // lanes 0-64 before the tile, 65-128 after it
    if (t <= 2 * kRadixRun) {
      const int64_t i = base - kRadixRun - 1 + hj;
      if (i >= 0 && i < n) halo = k1[i];
    }
#pragma unroll
    for (int r = 0; r < Items; ++r) s_key[1 + kRadixRun + r * kRadixFinishLanes + t] = raw[r];
    if (t <= 2 * kRadixRun) s_key[hj] = halo;
    __syncthreads();
    const auto tied = [&](int j) {
      const int64_t i = base - kRadixRun - 1 + j;
      return i > 0 && i < n && (R::canon(s_key[j]) >> low) == (R::canon(s_key[j - 1]) >> low);
    };
    for (int q = w; q < kRadixFinishTile / 64 + 2; q += NW) {
      const int j         = 1 + q * 64 + l;
      const bool tie      = tied(j);
      const uint64_t ties = __builtin_amdgcn_ballot_w64(tie);
      const uint64_t down = __builtin_amdgcn_ballot_w64(tie && R::canon(s_key[j]) < R::canon(s_key[j - 1]));
      if (l == 0) s_tied[q] = ties, s_down[q] = down;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < Items; ++r) {
      const int64_t i = base + r * kRadixFinishLanes + t;
      if (i >= n) break;
      const int j   = 1 + kRadixRun + r * kRadixFinishLanes + t;
      const int q   = w + r * NW;
      int64_t place = i;
      const uint64_t d1 = s_down[q + 1], d2 = s_down[q + 2];
      if (s_down[q] | d1 | d2) {
        // bits 0-2: this key and the two after it
        const uint64_t t1 = s_tied[q + 1], t2 = s_tied[q + 2];
        const unsigned tie  = unsigned((t1 >> l) | (l ? t2 << (64 - l) : 0)) & 7u;
        const unsigned down = unsigned((d1 >> l) | (l ? d2 << (64 - l) : 0)) & 3u;
        const bool tie_back = l ? ((t1 >> (l - 1)) & 1) != 0 : (s_tied[q] >> 63) != 0;
        if ((tie & 3u) == 0) {
          // no such neighbour
        } else if (tie == 2u) {  // the first of two
          place = i + (down >> 1);
        } else if ((tie & 3u) == 1u && !tie_back) {  // the second of two
          place = i - (down & 1u);
        } else {
          place = i + radix_place_in_run<R>(s_key, j, tied, broken);
        }
      }
      k0[place] = R::decode(raw[r]);
      if constexpr (Pairs) p0[place] = v[r];
    }
    __syncthreads();
  }
  if (broken) status[0] = 1, status[1] = uint32_t(low);
}

// Runs of at most 1024 x Items keys, each sorted by one block in LDS: every
// pass ranks the keys the lanes hold, places them in digit order in LDS and
// takes them back in that order.  One run is a whole sort, in place; more of
// them go to `out` and `pay_out`, encoded, for k_radix_merge.  Launch latency
// and the digits' chain of barriers bound it, about 2.5 us a digit at one key a
// lane and 5 at eight.
constexpr int kRadixSmallLanes = 1024;

template <class T, class PT, bool Iota, int Items, bool Whole>
__global__ __launch_bounds__(kRadixSmallLanes) void k_radix_small(typename RadixKey<T>::U* keys, PT* pay, const int all_n,
                                                                  typename RadixKey<T>::U* out, PT* pay_out) {
  using R              = RadixKey<T>;
  using U              = typename R::U;
  constexpr bool Pairs = !std::is_same<PT, NoPayload>::value;
  constexpr int NW     = kRadixSmallLanes / 64;
  constexpr int Run    = kRadixSmallLanes * Items;
  using Wide           = std::conditional_t<(Pairs && sizeof(PT) > sizeof(U)), uint64_t, U>;
  __shared__ Wide s_tile[Run];
  __shared__ uint32_t wcnt[NW][256];
  __shared__ uint32_t s_wave[4];
  __shared__ U s_and, s_or;
  const int first = Whole ? 0 : int(blockIdx.x) * Run;
  const int n     = Whole || all_n - first < Run ? all_n - first : Run;
  keys += first;
  if constexpr (Pairs) pay += first;
  U* key_tile  = reinterpret_cast<U*>(s_tile);
  PT* pay_tile = reinterpret_cast<PT*>(s_tile);
  const int t = threadIdx.x, w = t >> 6, l = t & 63;
  const int rounds = (n + kRadixSmallLanes - 1) / kRadixSmallLanes;  // of 64 keys per wavefront
  const int wfirst = w * 64 * rounds;
  if (t == 0) {
    s_and = ~U(0);
    s_or  = U(0);
  }
  __syncthreads();
  U u[Items], all = ~U(0), any = U(0);
  PT v[Pairs ? Items : 1];
  uint32_t slot[Items];
#pragma unroll
  for (int r = 0; r < Items; ++r) {
    const int i = wfirst + r * 64 + l;
    u[r]        = ~U(0);  // past the end: stays behind every key
    if (r < rounds && i < n) {
      u[r] = R::encode(keys[i]);
      all &= R::canon(u[r]);
      any |= R::canon(u[r]);
      if constexpr (Pairs) {
        if constexpr (Iota) v[r] = PT(first + i);
        else v[r] = pay[i];
      }
    }
  }
  atomicAnd(&s_and, all);
  atomicOr(&s_or, any);
  __syncthreads();
  const U varying = s_and ^ s_or;
  for (int p = 0; p < R::passes; ++p) {
    const int shift = 8 * p;
    if (((varying >> shift) & U(255)) == 0) continue;  // the same digit in every key
    for (int k = t; k < NW * 256; k += kRadixSmallLanes) (&wcnt[0][0])[k] = 0;
    __syncthreads();
    radix_rank<R>(u, slot, shift, wcnt[w], rounds);
    __syncthreads();
    uint32_t count = 0, wc[NW];
    if (t < 256) {
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        wc[q] = wcnt[q][t];
        count += wc[q];
      }
    }
    uint32_t at = radix_prefix256<NW>(count, s_wave);
    if (t < 256) {
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        wcnt[q][t] = at;
        at += wc[q];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < Items; ++r) {
      if (r < rounds) {
        slot[r] += wcnt[w][R::digit(u[r], shift)];
        key_tile[slot[r]] = u[r];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < Items; ++r)
      if (r < rounds) u[r] = key_tile[wfirst + r * 64 + l];
    if constexpr (Pairs) {
      __syncthreads();
#pragma unroll
      for (int r = 0; r < Items; ++r)
        if (r < rounds) pay_tile[slot[r]] = v[r];
      __syncthreads();
#pragma unroll
      for (int r = 0; r < Items; ++r)
        if (r < rounds) v[r] = pay_tile[wfirst + r * 64 + l];
    }
  }
#pragma unroll
  for (int r = 0; r < Items; ++r) {
    const int i = wfirst + r * 64 + l;
    if (r < rounds && i < n) {
      if constexpr (Whole) {
        keys[i] = R::decode(u[r]);
        if constexpr (Pairs) pay[i] = v[r];
      } else {
        out[first + i] = u[r];
        if constexpr (Pairs) pay_out[first + i] = v[r];
      }
    }
  }
}

// Places the keys of several sorted runs: a key's position is its own in its
// run and, for every other run, the number of keys there that go before it,
// those of earlier runs also where they are equal.  The searches' latency
// bounds it, so a block takes 64 keys only, neighbours in order that read the
// same lines, its wavefronts search different runs and each kRadixAbreast of
// them at once: 64 runs of 1024 (int64, 8-byte value) pairs take 79 us with
// their sort, 157 with one wavefront for all runs; 8 or 16 at once are no
// faster.
constexpr int kRadixAbreast    = 4;
constexpr int kRadixMergeWaves = 4;

template <class T, class PT, int Run>
__global__ __launch_bounds__(64 * kRadixMergeWaves) void k_radix_merge(const typename RadixKey<T>::U* in,
                                                                       const PT* pay_in, const int n,
                                                                       typename RadixKey<T>::U* keys, PT* pay) {
  using R = RadixKey<T>;
  using U = typename R::U;
  __shared__ int s_at[kRadixMergeWaves][64];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i    = int(blockIdx.x) * 64 + l;
  const int own  = int(blockIdx.x) / (Run / 64);
  const int runs = (n + Run - 1) / Run;
  const U u      = in[i < n ? i : n - 1];
  const U key    = R::canon(u);
  int at         = 0;
  for (int q = w; q < runs; q += kRadixAbreast * kRadixMergeWaves) {
    int pos[kRadixAbreast], len[kRadixAbreast];
#pragma unroll
    for (int c = 0; c < kRadixAbreast; ++c) {
      const int run = q + c * kRadixMergeWaves;
      pos[c]        = 0;
      len[c]        = run >= runs || run == own ? 0 : n - run * Run < Run ? n - run * Run : Run;
    }
    // the keys below pos go before, those from pos + 2 * step - 1 on do not
    for (int step = Run; step > 0; step >>= 1) {
#pragma unroll
      for (int c = 0; c < kRadixAbreast; ++c) {
        const int run = q + c * kRadixMergeWaves, k = pos[c] + step;
        if (k <= len[c]) {
          const U other = R::canon(in[run * Run + k - 1]);
          if (other < key || (other == key && run < own)) pos[c] = k;
        }
      }
    }
#pragma unroll
    for (int c = 0; c < kRadixAbreast; ++c) at += pos[c];
  }
  s_at[w][l] = at;
  __syncthreads();
  if (w > 0 || i >= n) return;
  at = i - own * Run;
#pragma unroll
  for (int q = 0; q < kRadixMergeWaves; ++q) at += s_at[q][l];
  keys[at] = R::decode(u);
  if constexpr (!std::is_same<PT, NoPayload>::value) pay[at] = pay_in[i];
}

// ------------------------------------------------------------------ host side
// Device memory of the sort, kept between calls and grown on demand: a fresh
// allocation per call costs more than the smaller sorts themselves and slows
// the kernels right after it.  `buf` holds the second copy of keys and
// payload and the segments' counts, `control` the fixed part.  Calls hold the
// mutex until their passes have run, so sorts on different instances take
// turns; Kokkos::finalize frees it.
struct RadixWorkspace {
  std::mutex mtx;
  void* buf             = nullptr;
  size_t bytes          = 0;
  RadixControl* control = nullptr;
  uint32_t* status      = nullptr;  // pinned host words that k_radix_finish reports to
  int turn              = 0;
  bool hooked           = false;
  // under the mutex
  void hook();
  void fit(size_t need);
};

inline RadixWorkspace& radix_workspace() {
  static RadixWorkspace w;
  return w;
}

// Where merged sorts keep their runs: several, as such sorts on different
// streams may well run side by side, and a device runs about four at once.
// A call holds one until its kernels have run.
struct RadixMergeSpace {
  std::mutex mtx;
  void* buf = nullptr;
};
constexpr int kRadixMergeSpaces = 4;
inline RadixMergeSpace* radix_merge_spaces() {
  static RadixMergeSpace s[kRadixMergeSpaces];
  return s;
}

inline void radix_workspace_release() {
  for (int q = 0; q < kRadixMergeSpaces; ++q) {
    RadixMergeSpace& s = radix_merge_spaces()[q];
    std::lock_guard<std::mutex> lock(s.mtx);
    if (s.buf) KKMX_SAFE_CALL(mx_free(s.buf, nullptr));
    s.buf = nullptr;
  }
  RadixWorkspace& w = radix_workspace();
  std::lock_guard<std::mutex> lock(w.mtx);
  if (w.buf) KKMX_SAFE_CALL(mx_free(w.buf, nullptr));
  if (w.control) KKMX_SAFE_CALL(mx_free(w.control, nullptr));
  if (w.status) KKMX_SAFE_CALL(mx_host_free(w.status));
  w.buf     = nullptr;
  w.control = nullptr;
  w.status  = nullptr;
  w.bytes   = 0;
  w.turn    = 0;
  w.hooked  = false;
}

inline void RadixWorkspace::hook() {
  if (!hooked) push_finalize_hook(&radix_workspace_release);
  hooked = true;
}

inline void RadixWorkspace::fit(size_t need) {
  if (bytes >= need) return;
  if (buf) KKMX_SAFE_CALL(mx_free(buf, nullptr));
  buf   = nullptr;
  bytes = 0;
  KKMX_SAFE_CALL(mx_malloc(&buf, need, nullptr));
  bytes = need;
}

template <class Unused = void>
__global__ void k_radix_control_init(RadixControl* c) {
  if (threadIdx.x < 2) c->summary[threadIdx.x] = {~0ull, 0ull};
  if (threadIdx.x == 2) c->trim = 0;
}

inline size_t radix_round(size_t bytes) { return (bytes + 255) & ~size_t(255); }

// Tile and resident blocks per CU of the scatter.  From kRadixLarge keys on,
// larger tiles make longer runs per digit: int32 keys, 2^28 of them, take
// 0.78 ms a pass with 8192-key tiles, 0.86 with 6144, 1.1 with 4096; (int64,
// 8-byte value) pairs, 3 M of them, 281 us all eight passes with 6144-key tiles, 303
// with 4096 and 474 with 8192, which no longer fit two blocks' registers.  Below,
// smaller tiles reach more CUs: 10^6 float64 keys take 159 us with 4096-key
// tiles, 172 with 6144, 186 with 8192.
template <class T, class PT, bool Large>
struct RadixShape {
  static constexpr int lanes  = 512;
  static constexpr int items  = !Large ? 8 : std::is_same<PT, NoPayload>::value ? 16 : 12;
  static constexpr int blocks = Large ? 2 : 4;
};
constexpr int64_t kRadixLarge = int64_t(1) << 21;

// The launches of one sort.
template <class T, class PT>
struct RadixRun {
  using U = typename RadixKey<T>::U;
  mx_stream_t stream;
  int64_t n, segment;
  int segments;
  U *k0, *k1;
  PT *p0, *p1;
  RadixControl* ctl;
  int turn;
  uint32_t* counts;

  // Digit 0's counts, and the AND and OR of all keys.
  template <bool Iota>
  void fold() {
    int p = 0, shift = 0;
    bool yes = true;
    mx_launch_kernel(reinterpret_cast<const void*>(&k_radix_count<T, Iota>), unsigned(segments), kRadixCountLanes, 0,
                     stream, p, shift, n, segment, k0, k1, ctl, turn, yes, counts);
  }
  template <bool Iota, class Shape>
  void passes(int first, int last) {
    bool no   = false;
    int shift = 0;
    for (int p = first; p < last; ++p) {
      if (p > 0 || sizeof(T) == 8)  // digit 0 of 4-byte keys is counted by the fold
        mx_launch_kernel(reinterpret_cast<const void*>(&k_radix_count<T, Iota>), unsigned(segments), kRadixCountLanes,
                         0, stream, p, shift, n, segment, k0, k1, ctl, turn, no, counts);
      bool summed = segments > kRadixDirect;
      if (summed)
        mx_launch_kernel(reinterpret_cast<const void*>(&k_radix_offsets<T, Iota>), 64, kRadixOffsetLanes, 0, stream, p,
                         ctl, turn, counts, segments);
      mx_launch_kernel(reinterpret_cast<const void*>(&k_radix_scatter<T, PT, Iota, Shape::lanes, Shape::items>),
                       unsigned(segments), Shape::lanes, 0, stream, p, shift, n, segment, k0, k1, p0, p1, ctl, turn,
                       counts, summed);
    }
  }
  void sample(bool allow) {
    mx_launch_kernel(reinterpret_cast<const void*>(&k_radix_sample<T>), 1, 1024, 0, stream, k0, n, ctl, turn, allow);
  }
  void finish(uint32_t* status, int cus) {
    const int64_t tiles = (n + kRadixFinishTile - 1) / kRadixFinishTile;
    mx_launch_kernel(reinterpret_cast<const void*>(&k_radix_finish<T, PT>), unsigned(tiles < 2 * cus ? tiles : 2 * cus),
                     kRadixFinishLanes, 0, stream, n, k0, k1, p0, p1, ctl, turn, status);
  }
};

// Places of the keys in runs of kRadixRun keys or more that share the digits
// from bit `low` on, in order; the keys are ordered by those.
template <class T>
struct RadixLongRunsF {
  using R = RadixKey<T>;
  using U = typename R::U;
  const U* keys;
  int64_t n;
  int low;
  uint32_t* places;
  KOKKOS_INLINE_FUNCTION U high(int64_t i) const { return R::canon(R::encode(keys[i])) >> low; }
  KOKKOS_INLINE_FUNCTION bool in_long_run(const int64_t i) const {
    const U mine = high(i);
    if ((i == 0 || high(i - 1) != mine) && (i + 1 >= n || high(i + 1) != mine)) return false;
    int64_t below = i >= kRadixRun ? i - kRadixRun : -1, first = i;  // the run's first key is above `below`
    while (first - below > 1) {
      const int64_t mid = below + (first - below) / 2;
      if (high(mid) == mine) first = mid;
      else below = mid;
    }
    return first + kRadixRun - 1 < n && high(first + kRadixRun - 1) == mine;
  }
  KOKKOS_INLINE_FUNCTION void operator()(const int64_t i, uint32_t& upd, const bool final) const {
    if (!in_long_run(i)) return;
    if (final) places[upd] = uint32_t(i);
    ++upd;
  }
};
// to[j] = from[places[j]], or back.
template <class U, class PT, bool Back>
struct RadixPlacesF {
  const uint32_t* places;
  const U* from;
  U* to;
  const PT* from_p;
  PT* to_p;
  KOKKOS_INLINE_FUNCTION void operator()(const int64_t j) const {
    const int64_t a = Back ? int64_t(places[j]) : j, b = Back ? j : int64_t(places[j]);
    to[a]           = from[b];
    if constexpr (!std::is_same<PT, NoPayload>::value) to_p[a] = from_p[b];
  }
};

// Whole tiles per segment and segments of n keys, as many as stay resident.
template <class Shape>
int radix_segments(int64_t n, int cus, int64_t& segment) {
  constexpr int tile   = Shape::lanes * Shape::items;
  const int64_t ntiles = (n + tile - 1) / tile;
  const int64_t tpb    = (ntiles + int64_t(cus) * Shape::blocks - 1) / (int64_t(cus) * Shape::blocks);
  segment              = tpb * tile;
  return int((ntiles + tpb - 1) / tpb);
}

template <class T, class PT, class Shape>
bool radix_sort_long_runs(const MI355X& exec, RadixWorkspace& ws, const RadixRun<T, PT>& r, int low, int cus);

// The passes of a sort that one block cannot hold.
template <class T, class PT, bool Iota, class Shape>
void radix_sort_passes(const MI355X& exec, typename RadixKey<T>::U* k0, int64_t n, PT* payload) {
  using U              = typename RadixKey<T>::U;
  constexpr bool pairs = !std::is_same<PT, NoPayload>::value;
  const int cus            = MI355X::impl_cu_count() > 0 ? MI355X::impl_cu_count() : 256;
  int64_t segment          = 0;
  const int segments       = radix_segments<Shape>(n, cus, segment);
  const size_t key_bytes   = radix_round(size_t(n) * sizeof(U));
  const size_t pay_bytes   = pairs ? radix_round(size_t(n) * sizeof(PT)) : 0;
  // counts for any number of keys: runs of some are sorted apart
  const size_t need        = key_bytes + pay_bytes + size_t(cus) * Shape::blocks * 256 * sizeof(uint32_t);
  RadixWorkspace& ws       = radix_workspace();
  std::lock_guard<std::mutex> lock(ws.mtx);
  ws.hook();
  ws.fit(need);
  if (!ws.control) {
    void* c = nullptr;
    KKMX_SAFE_CALL(mx_malloc(&c, sizeof(RadixControl), nullptr));
    ws.control = static_cast<RadixControl*>(c);
    mx_launch_kernel(reinterpret_cast<const void*>(&k_radix_control_init<>), 1, 64, 0, exec.stream(), ws.control);
  }
  if (!ws.status) {
    void* h = nullptr;
    KKMX_SAFE_CALL(mx_host_alloc(&h, 64));
    ws.status = static_cast<uint32_t*>(h);
  }
  RadixRun<T, PT> r{exec.stream(),
                    n,
                    segment,
                    segments,
                    k0,
                    static_cast<U*>(ws.buf),
                    payload,
                    pairs ? reinterpret_cast<PT*>(static_cast<char*>(ws.buf) + key_bytes) : nullptr,
                    ws.control,
                    ws.turn,
                    reinterpret_cast<uint32_t*>(static_cast<char*>(ws.buf) + key_bytes + pay_bytes)};
  ws.turn ^= 1;
  if constexpr (sizeof(T) == 4) {
    r.template fold<Iota>();
    r.template passes<Iota, Shape>(0, 4);
    // the workspace is free for the next call once the stream has run these
    exec.fence("Kokkos::sort: radix passes");
  } else {
    uint32_t* status = ws.status;
    *status          = 0;
    r.template fold<Iota>();
    r.sample(true);
    r.template passes<Iota, Shape>(0, kRadixTrim);
    r.finish(status, cus);
    exec.fence("Kokkos::sort: radix passes");
    if (*static_cast<volatile uint32_t*>(status) == 2) {
      r.template passes<Iota, Shape>(kRadixTrim, 8);
      exec.fence("Kokkos::sort: remaining radix passes");
    } else if (*static_cast<volatile uint32_t*>(status) == 1) {
      // the payload holds the permutation so far, also with Iota
      r.turn = ws.turn;
      if (radix_sort_long_runs<T, PT, Shape>(exec, ws, r, int(status[1]), cus)) return;
      ws.turn ^= 1;
      r.template fold<false>();
      r.sample(false);
      r.template passes<false, Shape>(0, 8);
      exec.fence("Kokkos::sort: all radix passes");
    }
  }
}

// One block sorts up to 16 KiB of keys.  Up to kRadixMerged keys are sorted in
// runs that k_radix_merge puts together, at most 24 of 1024 keys and then at
// most 24 of 4096; more keys go through the passes, which launch two or three
// kernels a digit but do not read every run for every key.  In us, one block /
// runs of 1024 / of 4096 / passes, int32 keys: 29 / 29 / 32 at 3000, 38 / 30 /
// 36 at 8192, runs 33 / 37 and passes 55 at 16384, 45 / 39 and 61 at 32768, 66 /
// 46 and 54 at 65536, 122 / 63 and 57 at 131072; (int64, 8-byte value) pairs:
// 37 / 37 / 39 at 1500, 43 / 37 / 45 at 3000, 65 / 38 / 54 at 8192, 43 / 53 and
// 94 at 16384, 55 / 56 and 100 at 32768, 79 / 65 and 94 at 65536, 143 / 84 and
// 98 at 131072, where pairs of few digits already gain from the passes.
template <class U>
constexpr int kRadixSmallItems    = sizeof(U) == 4 ? 4 : 2;
constexpr int kRadixMergeRuns     = 24;
constexpr int kRadixMerged        = kRadixMergeRuns * 4 * kRadixSmallLanes;
constexpr size_t kRadixMergeBytes = size_t(kRadixMerged) * 16;  // 8-byte keys and payload

// The launches of a sort of at most kRadixMerged keys, which are in order, and
// `space` free again, once the stream has run them.  `space` holds
// kRadixMergeBytes; one block's keys leave it alone.
template <class T, class PT, bool Iota>
void radix_sort_few(const MI355X& exec, typename RadixKey<T>::U* k0, int n, PT* payload, void* space) {
  using U = typename RadixKey<T>::U;
  U* k1   = static_cast<U*>(space);
  PT* p1  = nullptr;
  if constexpr (!std::is_same<PT, NoPayload>::value)
    p1 = reinterpret_cast<PT*>(static_cast<char*>(space) + kRadixMergeBytes / 2);
  const auto runs = [&](const void* sort, const void* merge, int run) {
    mx_launch_kernel(sort, unsigned((n + run - 1) / run), kRadixSmallLanes, 0, exec.stream(), k0, payload, n, k1, p1);
    mx_launch_kernel(merge, unsigned((n + 63) / 64), 64 * kRadixMergeWaves, 0, exec.stream(), k1, p1, n, k0, payload);
  };
  constexpr int R = kRadixSmallLanes;
  if (n <= R * kRadixSmallItems<U>)
    mx_launch_kernel(reinterpret_cast<const void*>(&k_radix_small<T, PT, Iota, kRadixSmallItems<U>, true>), 1, R, 0,
                     exec.stream(), k0, payload, n, k1, p1);
  else if (n <= kRadixMergeRuns * R)
    runs(reinterpret_cast<const void*>(&k_radix_small<T, PT, Iota, 1, false>),
         reinterpret_cast<const void*>(&k_radix_merge<T, PT, R>), R);
  else
    runs(reinterpret_cast<const void*>(&k_radix_small<T, PT, Iota, 4, false>),
         reinterpret_cast<const void*>(&k_radix_merge<T, PT, 4 * R>), 4 * R);
}

// The last step of a trimmed sort (`r`) with long runs out of order: their keys
// are sorted by all digits apart from the others and go back to the places that
// the runs had, which keeps the runs in order.  False, with nothing changed,
// where they are more than a fifth of all keys.  The second buffers hold the
// places, the runs' keys and payload and those sorts' second buffers.  3 M
// (int64, 8-byte) pairs with one such run of 300 take 323 us, where sorting all
// of them over by all digits made it 543, and 231 without the run; 2^25 int64
// keys 1.52 ms, 2.93 and 1.22.
template <class T, class PT, class Shape>
bool radix_sort_long_runs(const MI355X& exec, RadixWorkspace& ws, const RadixRun<T, PT>& r, int low, int cus) {
  using U              = typename RadixKey<T>::U;
  constexpr bool pairs = !std::is_same<PT, NoPayload>::value;
  using Range          = RangePolicy<MI355X, IndexType<int64_t>>;
  uint32_t* places     = reinterpret_cast<uint32_t*>(r.k1);  // n of them at most: half of the keys' second buffer
  uint32_t total       = 0;
  parallel_scan("Kokkos::sort::long_runs", Range(exec, 0, r.n), RadixLongRunsF<T>{r.k0, r.n, low, places}, total);
  const int64_t m = int64_t(total);
  if (m > r.n / 5) return false;
  RadixRun<T, PT> own = r;
  own.n               = m;
  own.segments        = radix_segments<Shape>(m, cus, own.segment);
  own.k0              = reinterpret_cast<U*>(reinterpret_cast<char*>(r.k1) + radix_round(size_t(r.n) * sizeof(uint32_t)));
  own.k1              = own.k0 + m;
  if constexpr (pairs) {
    own.p0 = r.p1;
    own.p1 = r.p1 + m;
  }
  parallel_for("Kokkos::sort::take_long_runs", Range(exec, 0, m),
               RadixPlacesF<U, PT, false>{places, r.k0, own.k0, r.p0, own.p0});
  if (m <= kRadixSmallLanes * kRadixSmallItems<U>) {
    radix_sort_few<T, PT, false>(exec, own.k0, int(m), own.p0, nullptr);
  } else {
    ws.turn ^= 1;  // r.turn is taken
    own.template fold<false>();
    own.sample(false);
    own.template passes<false, Shape>(0, 8);
  }
  parallel_for("Kokkos::sort::place_long_runs", Range(exec, 0, m),
               RadixPlacesF<U, PT, true>{places, own.k0, r.k0, own.p0, r.p0});
  exec.fence("Kokkos::sort: long runs");
  return true;
}

// A space for a merged sort, held until its owner is done with it.
inline void* radix_merge_space(std::unique_lock<std::mutex>& lock) {
  RadixMergeSpace* space = radix_merge_spaces();
  for (int q = 0; q < kRadixMergeSpaces && !lock.owns_lock(); ++q) {
    space = radix_merge_spaces() + q;
    lock  = std::unique_lock<std::mutex>(space->mtx, std::try_to_lock);
  }
  if (!lock.owns_lock()) lock.lock();
  if (!space->buf) {
    {
      std::lock_guard<std::mutex> hooks(radix_workspace().mtx);
      radix_workspace().hook();
    }
    KKMX_SAFE_CALL(mx_malloc(&space->buf, kRadixMergeBytes, nullptr));
  }
  return space->buf;
}

// Ascending LSD radix sort of n keys in place (device memory), on exec.
// With a payload (n device words of PT), the sort is of (key, payload)
// pairs and the payload is permuted with the keys, in place; with iota the
// payload's input is ignored and it receives the sorting permutation
// (sorted key i came from position payload[i]).
template <class T, class PT = NoPayload, bool Iota = false>
void radix_sort(const MI355X& exec, T* keys, int64_t n, PT* payload = nullptr) {
  static_assert(std::is_same<PT, NoPayload>::value || sizeof(PT) == 4 || sizeof(PT) == 8,
                "radix sort payloads are 4- or 8-byte words");
  static_assert(!Iota || std::is_same<PT, uint32_t>::value, "a permutation payload is 32-bit");
  if (n > int64_t(0x7fffffff)) throw_runtime_exception("Kokkos::sort: more than 2^31 - 1 keys");
  if (n < 1 || (n < 2 && !Iota)) return;
  using U = typename RadixKey<T>::U;
  U* k0   = reinterpret_cast<U*>(keys);
  if (n <= kRadixMerged) {
    std::unique_lock<std::mutex> lock;
    void* space = n <= kRadixSmallLanes * kRadixSmallItems<U> ? nullptr : radix_merge_space(lock);
    radix_sort_few<T, PT, Iota>(exec, k0, int(n), payload, space);
    exec.fence("Kokkos::sort: few keys");
    return;
  }
  if (n >= kRadixLarge) radix_sort_passes<T, PT, Iota, RadixShape<T, PT, true>>(exec, k0, n, payload);
  else radix_sort_passes<T, PT, Iota, RadixShape<T, PT, false>>(exec, k0, n, payload);
}

}  // namespace Impl
}  // namespace Kokkos

#endif
