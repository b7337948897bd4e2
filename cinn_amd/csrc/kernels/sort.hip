// argsort / sort along one axis: cinn_call_hip_argsort.
//
// What the reference computes (cinn/hlir/op/contrib/sort.cc:50-139 over the intrinsics cinn_host_lt_num_* /
// cinn_host_gt_num_* and cinn_host_next_smallest_int32, cinn/runtime/cpu/host_intrinsics.cc:67-106; the same on the GPU,
// cinn_cuda_runtime_source.cuh:645-715): every element gets the count of elements of its row that are smaller (larger
// when descending) - its *position* - and the index list is then built by taking, slot after slot, the element with
// the smallest position that has not been taken yet, the first such element on ties.  So the result is the order by
// (position, index): a stable sort, ascending or descending, with every NaN at position 0 (no comparison with a NaN
// is true) interleaved by index with the other elements of position 0.
//
// The reference's device code runs that second step from every thread on one shared buffer of positions that each
// call overwrites - it races.  Here an element computes its final slot directly:
//   slot(k) = #{ j : position(j) < position(k) } + #{ j < k : position(j) == position(k) },
// which is the same order and needs no shared mutable state; the index (and for sort the value) is scattered to that
// slot.  Rows without a NaN - the usual case, checked per tile - need one pass only, because position order is value
// order there: slot(k) = #{ x_j < x_k } + #{ j < k : x_j == x_k }.
//
// One block owns a tile of `size` elements along the sorted axis x TI neighbours along the axes after it (consecutive
// in memory, so loads and stores of a tile are whole lines when inner > 1; TI = 1 for the trailing axis).  The keys sit
// in LDS; the scan over a column reads four keys per instruction, the same for every lane of a column (a broadcast).
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>
#include <type_traits>

#include "cinn_hip_runtime.h"
#include "runtime/hip_check.h"

namespace {

constexpr int kThreads  = 256;
constexpr int kLdsLimit = 128 * 1024;

struct SortParams {
  const void* x;
  int32_t* index;  // may be null
  int32_t* rank;   // may be null: the position of every element (count of smaller / larger elements of its row)
  void* sorted;    // may be null
  int64_t* index64;  // may be null
  int size, inner, ti;  // ti: neighbouring columns per tile
  int keep;             // the first `keep` slots are written (the outputs' extent along the axis); ranks are for all elements
  int tiles_per_outer;  // ceil(inner / ti)
  int descending;
};

template <typename T>
struct KeyOf {
  typedef float type;
};
template <>
struct KeyOf<double> {
  typedef double type;
};
template <>
struct KeyOf<int32_t> {
  typedef int32_t type;
};
template <>
struct KeyOf<int64_t> {
  typedef int64_t type;
};

template <typename K>
__device__ __forceinline__ bool IsNan(K v) {
  return v != v;
}

// Ahead: a comes strictly before b in value order; AheadOrEqual: or ties with it
template <bool DESC, typename K>
__device__ __forceinline__ bool Ahead(K a, K b) {
  return DESC ? a > b : a < b;
}
template <bool DESC, typename K>
__device__ __forceinline__ bool AheadOrEqual(K a, K b) {
  return DESC ? a >= b : a <= b;
}

// a key that is never strictly ahead of any other: the padding of a column
template <bool DESC, typename K>
__device__ __forceinline__ K LastKey() {
  if (sizeof(K) == 8 && K(0.5) != K(0)) return DESC ? K(-__builtin_huge_val()) : K(__builtin_huge_val());
  if (K(0.5) != K(0)) return DESC ? K(-__builtin_huge_valf()) : K(__builtin_huge_valf());
  if (sizeof(K) == 8) return DESC ? K(LLONG_MIN) : K(LLONG_MAX);
  return DESC ? K(INT_MIN) : K(INT_MAX);
}

template <typename T, bool DESC>
__global__ void __launch_bounds__(kThreads) argsort_tile_kernel(SortParams p) {
  typedef typename KeyOf<T>::type K;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int size = p.size, ti = p.ti;
  const int size4 = (size + 3) & ~3;  // rows of the tile, padded so that four keys of a column are one aligned read
  K* const keys = reinterpret_cast<K*>(lds);                                   // [ti][size4]
  int* const pos = reinterpret_cast<int*>(lds + (size_t)ti * size4 * sizeof(K));  // [ti][size4], NaN tiles only
  const int outer = blockIdx.x / p.tiles_per_outer;
  const int i0    = (blockIdx.x - outer * p.tiles_per_outer) * ti;
  const int cols  = min(ti, p.inner - i0);
  const int64_t base = (int64_t)outer * size * p.inner + i0;
  const T* const X   = static_cast<const T*>(p.x);
  const int items    = size * cols;

  // item q = row k = q / cols, column c = q % cols: consecutive threads on consecutive addresses
  int has_nan = 0;
  for (int q = threadIdx.x; q < items; q += kThreads) {
    const int k = q / cols, c = q - k * cols;
    const K v   = static_cast<K>(X[base + (int64_t)k * p.inner + c]);
    keys[c * size4 + k] = v;
    has_nan |= IsNan(v) ? 1 : 0;
  }
  // the padding is read, four keys at a time, with the keys behind an element: never strictly ahead of anything
  for (int q = threadIdx.x; q < cols * (size4 - size); q += kThreads) {
    const int c = q / (size4 - size), k = size + q - c * (size4 - size);
    keys[c * size4 + k] = LastKey<DESC, K>();
  }
  has_nan = __syncthreads_or(has_nan);

  const int64_t result = (int64_t)outer * p.keep * p.inner + i0;
  auto scatter = [&](int k, int c, int slot, int position) {
    if (p.rank) p.rank[base + (int64_t)k * p.inner + c] = position;
    if (slot >= p.keep) return;
    const int64_t at = result + (int64_t)slot * p.inner + c;
    if (p.index) p.index[at] = k;
    if (p.index64) p.index64[at] = k;
    if (p.sorted) static_cast<T*>(p.sorted)[at] = X[base + (int64_t)k * p.inner + c];
  };

  if (!has_nan) {
    // here items are (column, row) with the row fastest: the lanes of a wavefront scan the same column.  Keys before
    // the element count when they are ahead of it or equal, keys behind it when they are strictly ahead: two loops of
    // one comparison and one add per key, around the group of four that holds the element itself.
    for (int q = threadIdx.x; q < items; q += kThreads) {
      const int c = q / size, k = q - c * size;
      const K* col = keys + c * size4;
      const K mine = col[k];
      const int kg = k & ~3;
      int slot = 0, ahead = 0;
      for (int j = 0; j < kg; j += 4) {
        K v[4];
        __builtin_memcpy(v, col + j, sizeof(v));
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          slot += AheadOrEqual<DESC>(v[u], mine) ? 1 : 0;
          ahead += Ahead<DESC>(v[u], mine) ? 1 : 0;
        }
      }
      {
        K v[4];
        __builtin_memcpy(v, col + kg, sizeof(v));
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const bool is_ahead = Ahead<DESC>(v[u], mine);
          ahead += is_ahead ? 1 : 0;
          slot += (is_ahead || (kg + u < k && v[u] == mine)) ? 1 : 0;
        }
      }
      int behind = 0;
      for (int j = kg + 4; j < size4; j += 4) {
        K v[4];
        __builtin_memcpy(v, col + j, sizeof(v));
#pragma unroll
        for (int u = 0; u < 4; ++u) behind += Ahead<DESC>(v[u], mine) ? 1 : 0;
      }
      scatter(k, c, slot + behind, ahead + behind);
    }
    return;
  }

  // tiles with a NaN: positions first, then the order by (position, index)
  for (int q = threadIdx.x; q < items; q += kThreads) {
    const int c = q / size, k = q - c * size;
    const K* col = keys + c * size4;
    const K mine = col[k];
    int ahead = 0;
    for (int j = 0; j < size; ++j) ahead += Ahead<DESC>(col[j], mine) ? 1 : 0;
    pos[c * size4 + k] = ahead;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < items; q += kThreads) {
    const int c = q / size, k = q - c * size;
    const int* col = pos + c * size4;
    const int mine = col[k];
    int slot = 0;
    for (int j = 0; j < size; ++j) slot += (col[j] < mine || (col[j] == mine && j < k)) ? 1 : 0;
    scatter(k, c, slot, mine);
  }
}

// ---- rows of 16- and 32-bit types ------------------------------------------------------------------------------------
// The scan above costs size^2 comparisons; these sort a row by (key, index), both in one 64-bit word: the key mapped to
// an unsigned number that grows in the wanted order (-0 and 0 alike, descending inverted), the index below it.  Distinct
// words, so any sorting network gives the stable order.  A NaN has position 0, i.e. it ties with the row's first
// element: its key becomes that element's.
template <typename T>
__device__ __forceinline__ uint32_t OrderedKey(T v, uint32_t invert, bool* is_nan) {
  const float f = static_cast<float>(v);
  *is_nan       = f != f;
  uint32_t u    = __builtin_bit_cast(uint32_t, f == 0.0f ? 0.0f : f);
  u ^= (u >> 31) ? 0xffffffffu : 0x80000000u;
  return u ^ invert;
}
template <>
__device__ __forceinline__ uint32_t OrderedKey<int32_t>(int32_t v, uint32_t invert, bool* is_nan) {
  *is_nan = false;
  return (static_cast<uint32_t>(v) ^ 0x80000000u) ^ invert;
}

typedef unsigned long long u64;
__device__ __forceinline__ u64 Word(uint32_t key, uint32_t index) { return ((u64)key << 32) | index; }

struct RowParams {
  const void* x;
  int32_t* index;    // argsort outputs, any may be null
  int32_t* rank;
  void* sorted;      // the first `keep` sorted values, any of these two may be null
  int64_t* index64;  // the first `keep` indices
  int size, inner, keep;
  uint32_t invert;   // 0xffffffff: descending
};

// the value of lane ^ X: within a row of 16 lanes on the vector ALU (DPP), across rows by the row swaps of gfx950
template <int X>
__device__ __forceinline__ uint32_t LaneXor(uint32_t v) {
  if constexpr (X == 1) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true);   // quad_perm [1,0,3,2]
  if constexpr (X == 2) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true);   // quad_perm [2,3,0,1]
  if constexpr (X == 4) return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 0x101F);                    // xor 4
  if constexpr (X == 8) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, true);  // row_ror 8
  if constexpr (X == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return threadIdx.x & 16 ? r[0] : r[1];
  }
  if constexpr (X == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return threadIdx.x & 32 ? r[0] : r[1];
  }
}
template <int X>
__device__ __forceinline__ u64 LaneXor64(u64 v) {
  return Word(LaneXor<X>((uint32_t)(v >> 32)), LaneXor<X>((uint32_t)v));
}
// minimum over a wavefront, the same in every lane
__device__ __forceinline__ uint32_t WaveMin32(uint32_t v) {
  v = min(v, LaneXor<1>(v));
  v = min(v, LaneXor<2>(v));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true));  // row_half_mirror: the other quad
  v = min(v, LaneXor<8>(v));
  v = min(v, LaneXor<16>(v));
  return min((uint32_t)__builtin_amdgcn_readlane((int)v, 0), (uint32_t)__builtin_amdgcn_readlane((int)v, 32));
}

// Block-wide reduction of a 32-bit number (only run for rows with a NaN).
template <int THREADS, typename F>
__device__ __forceinline__ uint32_t BlockReduce(uint32_t v, uint32_t* shared, F f) {
#pragma unroll
  for (int d = 1; d < 64; d *= 2) v = f(v, (uint32_t)__shfl_xor((int)v, d));
  if (THREADS == 64) return v;
  if ((threadIdx.x & 63) == 0) shared[threadIdx.x >> 6] = v;
  __syncthreads();
  v = shared[0];
#pragma unroll
  for (int w = 1; w < THREADS / 64; ++w) v = f(v, shared[w]);
  __syncthreads();
  return v;
}

// A thread's E words of its row, elements first + stride e; words beyond the row are larger than all others.  Returns the
// row's count of NaNs.
template <typename T, int E, int THREADS>
__device__ __forceinline__ int LoadWords(const RowParams& p, int64_t base, int first, int stride, int size, uint32_t* shared, u64 (&w)[E]) {
  const T* x = static_cast<const T*>(p.x) + base;
  uint32_t nans = 0, least = 0xffffffffu;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = first + stride * e;
    w[e]        = Word(0xffffffffu, (uint32_t)i);
    if (i < size) {
      bool nan;
      const uint32_t key = OrderedKey<T>(x[(int64_t)i * p.inner], p.invert, &nan);
      w[e] = Word(key, (uint32_t)i);
      if (nan) {
        nans |= 1u << e;
      } else {
        least = min(least, key);
      }
    }
  }
  const bool any = THREADS == 64 ? __any(nans != 0) : __syncthreads_or(nans != 0);
  if (!any) return 0;
  least = BlockReduce<THREADS>(least, shared, [](uint32_t a, uint32_t b) { return min(a, b); });
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (nans >> e & 1) w[e] = Word(least, (uint32_t)w[e]);
  return (int)BlockReduce<THREADS>(__popc(nans), shared, [](uint32_t a, uint32_t b) { return a + b; });
}

// One block sorts one row with a bitonic network over THREADS * E words: partners less than E apart are in one thread,
// less than 64 E apart in one wavefront (lane exchanges), the rest meet through LDS (3 of 55 layers at 1024 words).
// Bound by the 55 layers' vector instructions.  2048 rows of 1000 fp32 values, all three outputs: 229 -> 25 us against
// the scan; 16384 rows of 512 438 -> 133 us; columns, [32, 1000, 64] 687 -> 41 us.
template <typename T, int E, int THREADS>
__global__ void __launch_bounds__(THREADS) row_sort_kernel(RowParams p) {
  constexpr int N = E * THREADS;
  __shared__ u64 exchange[THREADS > 64 ? N : 1];
  __shared__ uint32_t shared[16];
  const int t        = threadIdx.x;
  const int64_t base = (int64_t)(blockIdx.x / p.inner) * p.size * p.inner + blockIdx.x % p.inner;
  u64 w[E];
  const int nans = LoadWords<T, E, THREADS>(p, base, t * E, 1, p.size, shared, w);
#pragma unroll 1
  for (int k = 2; k <= N; k *= 2) {
#pragma unroll 1
    for (int j = k / 2; j >= 64 * E; j /= 2) {
      if constexpr (THREADS > 64) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; ++e) exchange[e * THREADS + t] = w[e];
        __syncthreads();
        const int partner   = t ^ (j / E);
        const bool keep_min = ((t * E & j) == 0) == ((t * E & k) == 0);
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const u64 other = exchange[e * THREADS + partner];
          w[e]            = (other < w[e]) == keep_min ? other : w[e];
        }
      }
    }
    const bool up = (t * E & k) == 0;
    auto lanes = [&](auto distance) {
      constexpr int X = decltype(distance)::value;
      if (X * E >= k) return;
      const bool keep_min = ((t & X) == 0) == up;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const u64 other = LaneXor64<X>(w[e]);
        w[e]            = (other < w[e]) == keep_min ? other : w[e];
      }
    };
    lanes(std::integral_constant<int, 32>());
    lanes(std::integral_constant<int, 16>());
    lanes(std::integral_constant<int, 8>());
    lanes(std::integral_constant<int, 4>());
    lanes(std::integral_constant<int, 2>());
    lanes(std::integral_constant<int, 1>());
#pragma unroll
    for (int j = E / 2; j >= 1; j /= 2) {
      if (j < k) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          if ((e & j) != 0) continue;
          const bool up = ((t * E + e) & k) == 0;
          const u64 a = w[e], b = w[e | j];
          const bool swap = (b < a) == up;
          w[e]     = swap ? b : a;
          w[e | j] = swap ? a : b;
        }
      }
    }
  }
  const T* x = static_cast<const T*>(p.x) + base;
  const int64_t row = (int64_t)(blockIdx.x / p.inner) * p.keep * p.inner + blockIdx.x % p.inner;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int slot = t * E + e;
    const uint32_t i = (uint32_t)w[e];
    if (slot >= p.keep) continue;
    const int64_t at = row + (int64_t)slot * p.inner;
    if (p.index) p.index[at] = (int32_t)i;
    if (p.index64) p.index64[at] = (int64_t)i;
    if (p.sorted) static_cast<T*>(p.sorted)[at] = x[(int64_t)i * p.inner];
  }
  if (p.rank == nullptr) return;
  // The position of an element is the slot of the first element of equal key - a running maximum over the slots that
  // start a run - less the NaNs, which are no one's smaller element and all lie in the first run.
  uint32_t before = 0;
  {
    const uint32_t last = (uint32_t)(w[E - 1] >> 32);
    before = (uint32_t)__shfl_up((int)last, 1);
    if (THREADS > 64) {
      __syncthreads();
      if ((t & 63) == 63) shared[t >> 6] = last;
      __syncthreads();
      if ((t & 63) == 0 && t > 0) before = shared[(t >> 6) - 1];
    }
  }
  int head[E], run = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const uint32_t key = (uint32_t)(w[e] >> 32);
    if (key != before) run = t * E + e;
    head[e] = run;
    before  = key;
  }
  int upto = run;  // the last run start of the threads up to this one
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int v = __shfl_up(upto, d);
    if ((t & 63) >= d) upto = max(upto, v);
  }
  int earlier = __shfl_up(upto, 1);
  if ((t & 63) == 0) earlier = 0;
  if (THREADS > 64) {
    __syncthreads();
    if ((t & 63) == 63) shared[t >> 6] = (uint32_t)upto;
    __syncthreads();
    for (int v = 0; v < (t >> 6); ++v) earlier = max(earlier, (int)shared[v]);
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int start = max(head[e], earlier);
    if (t * E + e < p.size) p.rank[base + (int64_t)(uint32_t)w[e] * p.inner] = start > 0 ? start - nans : 0;
  }
}

// least 64-bit word of a wavefront, the same in every lane: the keys first, then the indices of those that have it
__device__ __forceinline__ u64 WaveMin(u64 v) {
  const uint32_t key = (uint32_t)(v >> 32), low = WaveMin32(key);
  return Word(low, WaveMin32(key == low ? (uint32_t)v : 0xffffffffu));
}

// The first `keep` (at most 64) of a wavefront's words, E per lane, written to first[0 .. keep - 1] in order.  The keep-th
// least of the lanes' least keys bounds the keys that can be among them, and few others lie below it: for the first five of
// 1000 random values seven words are left on average, for the first fifty about ninety.  These are gathered, C per lane, and
// each counts the ones before it.  Of the words at the bound itself the first `keep` suffice; that is looked at for C > 1 only.  (For
// C = 1 it takes rows of equal scores, 2048 of 1000, k = 5, from 9.5 to 6.2 us, where taking them one by one at once is 7.9, but is 0.1 to 0.3 us
// of every other row's time: k = 16 of 2048 rows of 200 4.9 -> 5.3.)  Should more than 64 C words be
// left - a lane has many of a row's first elements - they are taken one by one, the owner of each looking for its next one.
// candidates: 64 C words of LDS of this wavefront's own, as first is.  w[e] of a lane is ahead of w[e] of the lanes behind it
// and of all w[e + 1] where the keys are equal.
template <int E, int C>
__device__ __forceinline__ void SelectFirst(u64 (&w)[E], int keep, u64* candidates, u64* first) {
  const int lane = threadIdx.x & 63;
  uint32_t rest  = (uint32_t)(w[0] >> 32), limit = 0;
#pragma unroll
  for (int e = 1; e < E; ++e) rest = min(rest, (uint32_t)(w[e] >> 32));
#pragma unroll 1
  for (int s = 0; s < keep; ++s) {
    limit = WaveMin32(rest);
    if (lane == __builtin_ctzll(__ballot(rest == limit))) rest = 0xffffffffu;
  }
  const u64 before = ((u64)1 << lane) - 1;
  int count = 0, equals = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const uint32_t key = (uint32_t)(w[e] >> 32);
    u64 mask           = __ballot(C > 1 ? key < limit : key <= limit);
    if constexpr (C > 1) {
      const u64 equal = __ballot(key == limit);
      if (equal != 0 && equals < keep) {
        mask |= __ballot(key == limit && equals + __popcll(equal & before) < keep);
        equals += __popcll(equal);
      }
    }
    if (mask == 0) continue;
    const int at = count + __popcll(mask & before);
    if ((mask >> lane & 1) && at < 64 * C) candidates[at] = w[e];
    count += __popcll(mask);
  }
  if (count <= 64 * C) {
    // the wavefront's own words: its LDS accesses keep their order, the compiler must not change it
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
    u64 mine[C];
    int slot[C];
#pragma unroll
    for (int u = 0; u < C; ++u) mine[u] = lane + 64 * u < count ? candidates[lane + 64 * u] : ~0ull, slot[u] = 0;
#pragma unroll
    for (int v = 0; v < C; ++v) {
#pragma unroll 1
      for (int c = 0; c < min(count - 64 * v, 64); ++c) {
        const u64 other =
            Word((uint32_t)__builtin_amdgcn_readlane((int)(mine[v] >> 32), c), (uint32_t)__builtin_amdgcn_readlane((int)mine[v], c));
#pragma unroll
        for (int u = 0; u < C; ++u) slot[u] += other < mine[u] ? 1 : 0;
      }
    }
#pragma unroll
    for (int u = 0; u < C; ++u)
      if (lane + 64 * u < count && slot[u] < keep) first[slot[u]] = mine[u];
  } else {
    u64 least = w[0];
#pragma unroll
    for (int e = 1; e < E; ++e) least = w[e] < least ? w[e] : least;
#pragma unroll 1
    for (int s = 0; s < keep; ++s) {
      const u64 got = WaveMin(least);
      if (lane == s) first[s] = got;
      if (least == got) {
#pragma unroll
        for (int e = 0; e < E; ++e) w[e] = w[e] == got ? ~0ull : w[e];
        least = w[0];
#pragma unroll
        for (int e = 1; e < E; ++e) least = w[e] < least ? w[e] : least;
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// The first `keep` (at most kSelect) elements of a row.  A row of more than 1024 elements has several wavefronts; each selects
// the first `keep` of its part.  Of up to sixteen (C = 1) the first wavefront selects again, of more each looks up how many of
// the other parts' are before it.
// Bound by the launch and the read of the row for few elements (2048 rows of 1000 fp32 values in the last-level cache, k = 1: 5.6 us; an empty
// launch 3.3; rows from memory add 2.7, the one trip that all of a wavefront's work waits for), by the wave
// reductions that find the bound for many.  Taking the elements one by one - a 64-bit look at all of the owner's words for
// each - against this: k = 5 7.8 -> 6.3 us, k = 10 10.5 -> 7.0, k = 16 13.8 -> 7.9; 64 rows of 8000 fp16, k = 10 18.0 -> 8.7;
// 600 rows of 3000, k = 5 9.2 -> 6.5.
constexpr int kSelect = 64;  // what a wavefront can select
template <typename T, int E, int WAVES, int C>
__global__ void __launch_bounds__(64 * WAVES) row_select_kernel(RowParams p) {
  __shared__ u64 candidates[WAVES * 64 * C];
  __shared__ u64 part[WAVES][kSelect], first[WAVES > 1 && C == 1 ? 16 : 1];
  __shared__ uint32_t shared[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t base = (int64_t)(blockIdx.x / p.inner) * p.size * p.inner + blockIdx.x % p.inner;
  u64 w[E];
  LoadWords<T, E, 64 * WAVES>(p, base, t, 64 * WAVES, p.size, shared, w);
  SelectFirst<E, C>(w, p.keep, candidates + wave * 64 * C, part[wave]);
  if (WAVES > 1) __syncthreads();
  if constexpr (WAVES > 1 && C == 1) {
    if (wave > 0) return;
    u64 all[WAVES / 4];
#pragma unroll
    for (int e = 0; e < WAVES / 4; ++e) all[e] = (lane & 15) < p.keep ? part[e * 4 + (lane >> 4)][lane & 15] : ~0ull;
    SelectFirst<WAVES / 4, 1>(all, p.keep, candidates, first);
  }
  if (lane >= p.keep) return;
  const u64 mine = WAVES > 1 && C == 1 ? first[lane] : part[wave][lane];
  int slot       = lane;
  if constexpr (WAVES > 1 && C > 1) {
#pragma unroll 1
    for (int other = 0; other < WAVES; ++other) {
      if (other == wave) continue;
      int low = 0;  // words of the other part before this one: its list is in order
#pragma unroll
      for (int step = kSelect / 2; step > 0; step /= 2)
        if (low + step <= p.keep && part[other][low + step - 1] < mine) low += step;
      if (low < p.keep && part[other][low] < mine) ++low;
      slot += low;
    }
    if (slot >= p.keep) return;
  }
  const int64_t at = (int64_t)(blockIdx.x / p.inner) * p.keep * p.inner + blockIdx.x % p.inner + (int64_t)slot * p.inner;
  const uint32_t i = (uint32_t)mine;
  if (p.index64) p.index64[at] = (int64_t)i;
  if (p.sorted) static_cast<T*>(p.sorted)[at] = static_cast<const T*>(p.x)[base + (int64_t)i * p.inner];
}

// Columns (inner > 1) go to the network from this size: [32, 256, 64] 106 -> 16 us, [128, 256, 512] 679 -> 529 us (a
// column's accesses take a line each); at 64 elements the scan's whole-line tiles are ahead.
constexpr int kColumnSort   = 256;
// Short columns of which a good part is wanted go to the scan in top_k as well: a wavefront per column and a round per entry
// cost more.  us for k = 1 | 5 | 16, selection against scan, fp32: [1, 16, 100000] 27 | 54 | 139 against 14 | 14 | 16, [128, 64,
// 512] 25 | 38 | 96 against 66; [32, 100, 1000] 21 | 25 | 53 against 79.
constexpr int kColumnScan   = 64;
constexpr int kRowSortLimit = 16384;  // words of a row in one block's LDS (128 KiB)

template <typename T>
void LaunchRowSort(const RowParams& p, int rows, hipStream_t stream) {
#define CINN_ROW_SORT(E, THREADS) hipLaunchKernelGGL((row_sort_kernel<T, E, THREADS>), dim3(rows), dim3(THREADS), 0, stream, p)
  if (p.size <= 64) {
    CINN_ROW_SORT(1, 64);
  } else if (p.size <= 256) {
    CINN_ROW_SORT(4, 64);
  } else if (p.size <= 1024) {
    CINN_ROW_SORT(4, 256);
  } else if (p.size <= 4096) {
    CINN_ROW_SORT(4, 1024);
  } else {
    CINN_ROW_SORT(16, 1024);
  }
#undef CINN_ROW_SORT
}
template <typename T>
void LaunchRowSelect(const RowParams& p, int rows, hipStream_t stream) {
  // words per lane for what is left of a selection: 16 of 64 lanes' least ones bound about 20 words of 1000, 32 about 45 and
  // 50 about 90, with a spread that takes the last over 128 in a few rows of a hundred
#define CINN_ROW_SELECT_C(E, WAVES, C) \
  hipLaunchKernelGGL((row_select_kernel<T, E, WAVES, C>), dim3(rows), dim3(64 * WAVES), 0, stream, p)
#define CINN_ROW_SELECT(E, WAVES)      \
  if (p.keep <= 16) {                  \
    CINN_ROW_SELECT_C(E, WAVES, 1);    \
  } else if (p.keep <= 32) {           \
    CINN_ROW_SELECT_C(E, WAVES, 2);    \
  } else {                             \
    CINN_ROW_SELECT_C(E, WAVES, 4);    \
  }
  if (p.size <= 256) {
    CINN_ROW_SELECT(4, 1);
  } else if (p.size <= 1024) {
    CINN_ROW_SELECT(16, 1);
  } else if (p.size <= 4096) {
    CINN_ROW_SELECT(16, 4);
  } else {
    CINN_ROW_SELECT(16, 16);
  }
#undef CINN_ROW_SELECT
#undef CINN_ROW_SELECT_C
}

// Up to which k the selection is ahead of the network.  The network's time is the blocks per CU (four wavefronts for 257 to
// 1024 words, sixteen above), the selection's the chain of one wavefront, which grows with k and with the words up to the bound.
// us, network | selection, fp32: up to 256 rows of 400, k = 24 8.9 | 7.4, k = 32 8.9 | 8.9, k = 50 8.9 | 14; of 1000, k = 20 9.1 | 8.3, k =
// 24 9.1 | 8.9, k = 50 9.1 | 16.4; 600 rows of 1000, k = 32 11.7 | 10.7; 1024 of 400, k = 40 13.8 | 12.1, k = 50 13.2 | 15.2; 1500 of 400, k = 50
// 17.8 | 16.1; 2048 of 1000, k = 50 22.6 | 18.3.  (Where many scores are equal, rounded to halves, the selection takes a seventh more:
// 256 rows of 1000, k = 24 9.1 | 10.2, 1500, k = 50 18.4 | 20.8.)  64 rows of 1500, k = 50 18.4 | 16.1, of 4000 18.9 | 18.6 (with equal
// ones 18.9 | 19.9); 64 rows of 8000 fp16, k = 50 77.9 | 28.4; k = 64 of 600 rows of 1500 41.2 | 59 (with as many elements as lanes the
// bound is the largest of the lanes' least words, and most rows are taken one by one).  The network of 256 words on one wavefront
// is short: 4000 rows of 250, k = 17 9.5, k = 50 9.7 | 17.0.
int SelectLimit(int size, int rows) {
  if (size <= 256) return 16;
  const int per_cu = (rows + 255) / 256;  // the network's blocks
  if (size > 1024 || per_cu >= 8) return 50;
  static constexpr int kWide[8] = {0, 20, 24, 32, 32, 40, 40, 40}, kNarrow[8] = {0, 24, 32, 32, 40, 40, 50, 50};
  return size <= 768 ? kNarrow[per_cu] : kWide[per_cu];
}

enum class Elem { kF32, kF64, kF16, kBF16, kI32, kI64, kUnsupported };

Elem ElemOf(const cinn_buffer_t* b) {
  const auto& t = b->type;
  if (t.code == cinn_type_float && t.bits == 32) return Elem::kF32;
  if (t.code == cinn_type_float && t.bits == 64) return Elem::kF64;
  if (t.code == cinn_type_float && t.bits == 16) return Elem::kF16;
  if (t.code == cinn_type_bfloat && t.bits == 16) return Elem::kBF16;
  if (t.code == cinn_type_int && t.bits == 32) return Elem::kI32;
  if (t.code == cinn_type_int && t.bits == 64) return Elem::kI64;
  return Elem::kUnsupported;
}

cinn_buffer_t* BufferArg(void* v_args, int index) {
  auto* args = static_cast<cinn_pod_value_t*>(v_args);
  CINN_RT_CHECK(args[index].type_code_ == CINN_POD_BUFFER_P, "argsort: argument %d is not a buffer", index);
  auto* b = static_cast<cinn_buffer_t*>(args[index].value_.v_handle);
  CINN_RT_CHECK(b && b->memory, "argsort: argument %d has no device memory", index);
  return b;
}

template <typename T, bool DESC>
void LaunchDirection(const SortParams& p, int blocks, size_t lds_bytes, hipStream_t stream) {
  auto kernel = argsort_tile_kernel<T, DESC>;
  static const bool configured = [&] {  // once per instantiation, thread-safe
    CINN_HIP_CALL(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsLimit));
    return true;
  }();
  (void)configured;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kThreads), lds_bytes, stream, p);
}

template <typename T>
void Launch(const SortParams& p, int blocks, size_t lds_bytes, hipStream_t stream) {
  if (p.descending) {
    LaunchDirection<T, true>(p, blocks, lds_bytes, stream);
  } else {
    LaunchDirection<T, false>(p, blocks, lds_bytes, stream);
  }
}

// the scan: tiles of neighbouring columns
void LaunchTiles(SortParams p, Elem elem, int outer, hipStream_t s) {
  const size_t key_bytes = (elem == Elem::kF64 || elem == Elem::kI64) ? 8 : 4;
  const size_t per_col   = (size_t)((p.size + 3) & ~3) * (key_bytes + 4);  // keys and, for tiles with a NaN, positions
  CINN_RT_CHECK(per_col <= (size_t)kLdsLimit, "argsort: %d elements along the sorted axis exceed the %zu that one block's LDS holds", p.size,
                (size_t)kLdsLimit / (key_bytes + 4));
  // neighbouring columns per tile: whole 64-byte pieces of a row when there are that many, bounded by LDS and by the
  // work one block should carry
  int ti = p.inner < 16 ? p.inner : 16;
  while (ti > 1 && (per_col * ti > (size_t)kLdsLimit / 2 || (int64_t)p.size * ti > 8192)) ti /= 2;
  p.ti              = ti;
  p.tiles_per_outer = (p.inner + ti - 1) / ti;
  const int64_t blocks = (int64_t)outer * p.tiles_per_outer;
  CINN_RT_CHECK(blocks < INT_MAX, "argsort: too many tiles");
  const size_t lds_bytes = per_col * ti;
  switch (elem) {
    case Elem::kF32: Launch<float>(p, (int)blocks, lds_bytes, s); break;
    case Elem::kF64: Launch<double>(p, (int)blocks, lds_bytes, s); break;
    case Elem::kF16: Launch<_Float16>(p, (int)blocks, lds_bytes, s); break;
    case Elem::kBF16: Launch<__bf16>(p, (int)blocks, lds_bytes, s); break;
    case Elem::kI32: Launch<int32_t>(p, (int)blocks, lds_bytes, s); break;
    case Elem::kI64: Launch<int64_t>(p, (int)blocks, lds_bytes, s); break;
    default: break;
  }
  CINN_HIP_CALL(hipGetLastError());
}

}  // namespace

extern "C" void cinn_call_hip_argsort(void* v_args, int num_args, int outer, int size, int inner, int is_ascend,
                                       int outputs, void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  const int want = ((outputs & 1) ? 1 : 0) + ((outputs & 2) ? 1 : 0) + ((outputs & 4) ? 1 : 0);
  CINN_RT_CHECK(outputs >= 1 && outputs <= 7, "argsort: outputs is a set of bits 1 (indices), 2 (positions), 4 (sorted values), got %d", outputs);
  CINN_RT_CHECK(num_args == 1 + want, "argsort: the input and %d outputs expected, got %d arguments", want, num_args);
  CINN_RT_CHECK(outer >= 0 && size >= 0 && inner >= 0, "argsort: negative extent");
  if ((int64_t)outer * size * inner == 0) return;
  CINN_RT_CHECK((int64_t)outer * size * inner < INT_MAX, "argsort: tensor too large for 32-bit offsets");
  cinn_buffer_t* x = BufferArg(v_args, 0);
  const Elem elem  = ElemOf(x);
  CINN_RT_CHECK(elem != Elem::kUnsupported, "argsort: element type (code %d, %d bits) is not one of fp16 / bf16 / fp32 / fp64 / int32 / int64",
                (int)x->type.code, (int)x->type.bits);
  SortParams p{};
  p.x   = x->memory;
  int a = 1;
  auto int32_output = [&](const char* what) {
    cinn_buffer_t* b = BufferArg(v_args, a++);
    CINN_RT_CHECK(b->type.code == cinn_type_int && b->type.bits == 32, "argsort: the %s output must be int32", what);
    return reinterpret_cast<int32_t*>(b->memory);
  };
  if (outputs & 1) p.index = int32_output("index");
  if (outputs & 2) p.rank = int32_output("position");
  if (outputs & 4) {
    cinn_buffer_t* b = BufferArg(v_args, a++);
    CINN_RT_CHECK(b->type.code == x->type.code && b->type.bits == x->type.bits, "argsort: the sorted output must have the input's type");
    CINN_RT_CHECK(b->memory != x->memory, "argsort: sorting in place is not supported");
    p.sorted = b->memory;
  }
  p.size = p.keep = size, p.inner = inner, p.descending = is_ascend ? 0 : 1;
  auto s = static_cast<hipStream_t>(stream);
  // Rows of the trailing axis sort in a network; columns too once the scan's work outweighs its whole-line accesses.
  if (elem != Elem::kF64 && elem != Elem::kI64 && size <= kRowSortLimit && (inner == 1 || size >= kColumnSort)) {
    RowParams r{p.x, p.index, p.rank, p.sorted, nullptr, size, inner, size, is_ascend ? 0u : 0xffffffffu};
    switch (elem) {
      case Elem::kF32: LaunchRowSort<float>(r, outer * inner, s); break;
      case Elem::kF16: LaunchRowSort<_Float16>(r, outer * inner, s); break;
      case Elem::kBF16: LaunchRowSort<__bf16>(r, outer * inner, s); break;
      default: LaunchRowSort<int32_t>(r, outer * inner, s); break;
    }
    CINN_HIP_CALL(hipGetLastError());
    return;
  }
  LaunchTiles(p, elem, outer, s);
}

// The first k entries along an axis of the order cinn_call_hip_argsort gives: values (bit 1 of `outputs`) and int64
// indices (bit 2), each [outer][k][inner].
extern "C" void cinn_call_hip_top_k(void* v_args, int num_args, int outer, int size, int inner, int is_ascend, int k, int outputs,
                                     void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  CINN_RT_CHECK(outputs >= 1 && outputs <= 3, "top_k: outputs is a set of bits 1 (values), 2 (indices), got %d", outputs);
  const int want = (outputs & 1) + (outputs >> 1);
  CINN_RT_CHECK(num_args == 1 + want, "top_k: the input and %d outputs expected, got %d arguments", want, num_args);
  CINN_RT_CHECK(outer >= 0 && size >= 0 && inner >= 0, "top_k: negative extent");
  if ((int64_t)outer * size * inner == 0) return;
  CINN_RT_CHECK((int64_t)outer * size * inner < INT_MAX, "top_k: tensor too large for 32-bit offsets");
  CINN_RT_CHECK(k >= 1 && k <= size, "top_k: k = %d of %d elements", k, size);
  CINN_RT_CHECK(size <= kRowSortLimit, "top_k: %d elements along the axis, at most %d are supported", size, kRowSortLimit);
  cinn_buffer_t* x = BufferArg(v_args, 0);
  RowParams r{x->memory, nullptr, nullptr, nullptr, nullptr, size, inner, k, is_ascend ? 0u : 0xffffffffu};
  if (outputs & 1) {
    cinn_buffer_t* b = BufferArg(v_args, 1);
    CINN_RT_CHECK(b->type.code == x->type.code && b->type.bits == x->type.bits, "top_k: the values must have the input's type");
    r.sorted = b->memory;
  }
  if (outputs & 2) {
    cinn_buffer_t* b = BufferArg(v_args, num_args - 1);
    CINN_RT_CHECK(b->type.code == cinn_type_int && b->type.bits == 64, "top_k: the indices must be int64");
    r.index64 = reinterpret_cast<int64_t*>(b->memory);
  }
  auto s          = static_cast<hipStream_t>(stream);
  const Elem elem = ElemOf(x);
  if (inner > 1 && size <= kColumnScan && size <= 4 * k + 16 && elem != Elem::kF64 && elem != Elem::kI64 && elem != Elem::kUnsupported) {
    SortParams p{};
    p.x = r.x, p.sorted = r.sorted, p.index64 = r.index64;
    p.size = size, p.keep = k, p.inner = inner, p.descending = is_ascend ? 0 : 1;
    LaunchTiles(p, elem, outer, s);
    return;
  }
  auto run = [&](auto launch_select, auto launch_sort) { k <= SelectLimit(size, outer * inner) ? launch_select(r, outer * inner, s) : launch_sort(r, outer * inner, s); };
  switch (elem) {
    case Elem::kF32: run(LaunchRowSelect<float>, LaunchRowSort<float>); break;
    case Elem::kF16: run(LaunchRowSelect<_Float16>, LaunchRowSort<_Float16>); break;
    case Elem::kBF16: run(LaunchRowSelect<__bf16>, LaunchRowSort<__bf16>); break;
    case Elem::kI32: run(LaunchRowSelect<int32_t>, LaunchRowSort<int32_t>); break;
    default:
      CINN_RT_CHECK(false, "top_k: element type (code %d, %d bits) is not one of fp16 / bf16 / fp32 / int32", (int)x->type.code,
                    (int)x->type.bits);
  }
  CINN_HIP_CALL(hipGetLastError());
}
