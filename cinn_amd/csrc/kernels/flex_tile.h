// Device code shared by the register-staged MFMA kernels (gemm_flex.hip, conv_backward_mfma.hip): operand tiles on their
// way global -> registers -> LDS, the MFMAs of a K step, the pipelined K loop and the staging of the result tile.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace cinn_hip_kernels {
namespace flex {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// 16 bytes from any element-aligned address (one global_load_dwordx4: unaligned access is on for this target)
template <typename T>
__device__ __forceinline__ u32x4 LoadAny(const char* p) {
  u32x4 v;
  __builtin_memcpy(&v, __builtin_assume_aligned(p, sizeof(T)), 16);
  return v;
}

// One operand's ROWS x (K step) tile of a block.  KC: memory is [row][k], LDS [row][128 bytes].  Otherwise memory is
// [k][row], LDS [k][ROWS].
//
// LDS placement.  [row][128 B]: chunk c of a row lies at c ^ (row & 7) ^ ((row >> 3) & 1), which spreads the sixteen
// lanes a 16-byte fragment read serves together over sixteen bank groups.  [k][ROWS], 16-bit: a transposing read
// touches four k rows x two chunks per group of 16 lanes, two groups (k and k + 16) together; the keys below send those
// sixteen chunks to different bank groups.  [k][ROWS], 32-bit: the two halves of a wavefront read rows four apart, bit
// 2 of k flips the half of a 256-byte line.
template <typename T, bool KC, int ROWS, int THREADS>
struct Tile {
  static constexpr int E      = 16 / (int)sizeof(T);  // elements per chunk
  static constexpr int KS     = 8 * E;                // elements of a K step
  static constexpr int CHUNKS = ROWS * 8 / THREADS;   // chunks per thread and step
  static constexpr int CH     = ROWS / E;             // chunks per k row (not KC)

  const char* base;       // the tile's first element at k = 0
  int64_t step_bytes;     // along K
  unsigned off[CHUNKS];   // byte offset of the thread's chunks at step 0
  const char* end;        // end of the operand
  int rows_left;          // valid rows from the tile's first one

  static __device__ __forceinline__ int ChunkK(int tid, int i) { return KC ? (tid & 7) * E : tid / CH + i * (THREADS / CH); }
  static __device__ __forceinline__ int LdsOffset(int tid, int i) {
    if (KC) {
      const int row = (tid >> 3) + THREADS / 8 * i;
      return row * 128 + (((tid & 7) ^ (row & 7) ^ ((row >> 3) & 1)) << 4);
    }
    return RowOffset(ChunkK(tid, i), tid % CH);
  }
  // byte offset of chunk `c` of k row `k` ([k][ROWS] form)
  static __device__ __forceinline__ int RowOffset(int k, int c) {
    if (sizeof(T) == 4) return k * (ROWS * 4) + ((c ^ (((k >> 2) & 1) << 3)) << 4);
    if (ROWS == 128) return k * 256 + ((c ^ (2 * (k & 3)) ^ (8 * ((k >> 4) & 1))) << 4);
    return (k >> 1) * 256 + (((((k & 1) << 3) | c) ^ (((k >> 1) & 1) << 1) ^ (((k >> 4) & 1) << 2)) << 4);
  }

  __device__ __forceinline__ void Init(const void* p, int64_t ld, int row0, int rows, int k_total, int tid) {
    const char* q = static_cast<const char*>(p);
    rows_left     = rows - row0;
    if (KC) {
      base       = q + (int64_t)row0 * ld * sizeof(T);
      step_bytes = KS * sizeof(T);
      end        = nullptr;
#pragma unroll
      for (int i = 0; i < CHUNKS; ++i) {
        const int row = min((tid >> 3) + THREADS / 8 * i, rows_left - 1);
        off[i]        = (unsigned)(((int64_t)row * ld + ChunkK(tid, i)) * sizeof(T));
      }
    } else {
      base       = q + (int64_t)row0 * sizeof(T);
      step_bytes = (int64_t)KS * ld * sizeof(T);
      end        = q + ((int64_t)(k_total - 1) * ld + rows) * sizeof(T);
      const int first = min(tid % CH, (rows_left - 1) / E) * E;  // a chunk beyond the rows repeats the last one
#pragma unroll
      for (int i = 0; i < CHUNKS; ++i) off[i] = (unsigned)(((int64_t)ChunkK(tid, i) * ld + first) * sizeof(T));
    }
  }

  template <bool GUARD>
  __device__ __forceinline__ void Load(u32x4 (&r)[CHUNKS], int step, int k_total, int tid) const {
    const char* at = base + step * step_bytes;
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      if (!GUARD) {
        r[i] = LoadAny<T>(at + off[i]);
        continue;
      }
      const int k_left = k_total - step * KS - ChunkK(tid, i);  // valid k from the chunk's first one
      const char* p    = at + off[i];
      u32x4 v          = {0, 0, 0, 0};
      if (KC ? k_left >= E : (k_left > 0 && p + 16 <= end)) {
        v = LoadAny<T>(p);
      } else if (k_left > 0) {
        typedef T chunk_t __attribute__((ext_vector_type(E)));
        chunk_t part    = {0};
        const int first = KC ? 0 : min(tid % CH, (rows_left - 1) / E) * E;
        const int count = KC ? k_left : rows_left - first;
#pragma unroll
        for (int e = 0; e < E; ++e)
          if (e < count) part[e] = reinterpret_cast<const T*>(p)[e];
        v = __builtin_bit_cast(u32x4, part);
      }
      r[i] = v;
    }
  }
  __device__ __forceinline__ void Store(char* tile, const u32x4 (&r)[CHUNKS], int tid) const {
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) *reinterpret_cast<u32x4*>(tile + LdsOffset(tid, i)) = r[i];
  }
};

template <typename T>
struct Half16;
template <>
struct Half16<__bf16> {
  typedef bf16x8 vec8;
  static __device__ __forceinline__ f32x4 mfma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Half16<_Float16> {
  typedef f16x8 vec8;
  static __device__ __forceinline__ f32x4 mfma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// The MFMA work of one K step on a wavefront's WM x WN part of the block tile, and where its results lie.
template <typename T, bool A_KC, bool B_KC, int BM, int BN>
struct Mma {
  static constexpr int TM = BM / 2 / 16, TN = BN / 2 / 16;
  typedef f32x4 acc_t[TM][TN];
  typedef typename Half16<T>::vec8 vec8;

  static __device__ __forceinline__ void Zero(acc_t& acc) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  // v_mfma_f32_16x16x32: lane l holds row (column) l % 16 and eight consecutive k; the lane groups 0..3 take the k
  // chunks 0, 2, 1, 3 in either operand (which is free as long as both agree)
  template <bool KC, int ROWS>
  static __device__ __forceinline__ vec8 Fragment(const char* tile, int row0, int kk, int lane) {
    const int kg = ((lane >> 4) & 1) * 2 + (lane >> 5);
    if (KC) {
      const int row = row0 + (lane & 15);
      return *reinterpret_cast<const vec8*>(tile + row * 128 + (((kk * 4 + kg) ^ (row & 7) ^ ((row >> 3) & 1)) << 4));
    }
    s16x4 part[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int k = kk * 32 + 8 * kg + 4 * r + ((lane & 15) >> 2);
      const int n = row0 + 4 * (lane & 3);
      const char* p = tile + Tile<T, false, ROWS, 256>::RowOffset(k, n >> 3) + (n & 7) * 2;
      part[r] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)p);
    }
    return __builtin_bit_cast(vec8, __builtin_shufflevector(part[0], part[1], 0, 1, 2, 3, 4, 5, 6, 7));
  }
  template <int KG>
  static __device__ __forceinline__ void Step(const char* a_tile, const char* b_tile, int wm, int wn, int kg, int lane, acc_t& acc) {
#pragma unroll
    for (int part = 0; part < 2 / KG; ++part) {
      const int kk = kg * (2 / KG) + part;
      vec8 a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = Fragment<A_KC, BM>(a_tile, wm * (BM / 2) + i * 16, kk, lane);
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j] = Fragment<B_KC, BN>(b_tile, wn * (BN / 2) + j * 16, kk, lane);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = Half16<T>::mfma(a[i], b[j], acc[i][j]);
    }
  }
  // f(row, column, value) for every result of the wavefront, relative to its part of the tile
  template <typename F>
  static __device__ __forceinline__ void Each(const acc_t& acc, int lane, F f) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) f(i * 16 + 4 * (lane >> 4) + r, j * 16 + (lane & 15), acc[i][j][r]);
  }
};

template <bool A_KC, bool B_KC, int BM, int BN>
struct Mma<float, A_KC, B_KC, BM, BN> {
  static constexpr int TM = BM / 2 / 32, TN = BN / 2 / 32;
  typedef f32x16 acc_t[TM][TN];

  static __device__ __forceinline__ void Zero(acc_t& acc) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  }
  static __device__ __forceinline__ void Add(acc_t& acc, const acc_t& more) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] += more[i][j];
  }
  // four k of one row: chunk 2 q + (lane / 32), element e feeds MFMA (q, e) of v_mfma_f32_32x32x2_f32
  template <bool KC, int ROWS>
  static __device__ __forceinline__ f32x4 Fragment(const char* tile, int row0, int q, int lane) {
    const int row = row0 + (lane & 31), c = 2 * q + (lane >> 5);
    if (KC) return *reinterpret_cast<const f32x4*>(tile + row * 128 + ((c ^ (row & 7) ^ ((row >> 3) & 1)) << 4));
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = *reinterpret_cast<const float*>(tile + Tile<float, false, ROWS, 256>::RowOffset(4 * c + e, row >> 2) + (row & 3) * 4);
    return v;
  }
  template <int KG>
  static __device__ __forceinline__ void Step(const char* a_tile, const char* b_tile, int wm, int wn, int kg, int lane, acc_t& acc) {
#pragma unroll
    for (int part = 0; part < 4 / KG; ++part) {
      const int q = kg * (4 / KG) + part;
      f32x4 a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = Fragment<A_KC, BM>(a_tile, wm * (BM / 2) + i * 32, q, lane);
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j] = Fragment<B_KC, BN>(b_tile, wn * (BN / 2) + j * 32, q, lane);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
    }
  }
  template <typename F>
  static __device__ __forceinline__ void Each(const acc_t& acc, int lane, F f) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) f(i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), j * 32 + (lane & 31), acc[i][j][r]);
  }
};

// Consecutive block ids go round-robin to the 8 XCDs, each with its own L2: every XCD gets a contiguous run of tiles,
// walked down eight tile rows before the next tile column, so that its blocks share operand panels.
__device__ __forceinline__ void TileOf(int bid, int tiles_m, int tiles_n, int* tm, int* tn) {
  const int tiles = tiles_m * tiles_n;
  const int q = tiles >> 3, r = tiles & 7, xcd = bid & 7;
  const int id    = xcd * q + min(xcd, r) + (bid >> 3);
  const int width = 8 * tiles_n, group = id / width, first = group * 8;
  const int rows = min(tiles_m - first, 8), in = id - group * width;
  *tm = first + in % rows;
  *tn = in / rows;
}

// A K step whose products are summed in PARTS chains of their own before they are added to acc.
template <typename M, int PARTS>
__device__ __forceinline__ void InParts(const char* a_tile, const char* b_tile, int wm, int wn, int lane, typename M::acc_t& acc) {
  typename M::acc_t sum[PARTS];
#pragma unroll
  for (int part = 0; part < PARTS; ++part) {
    M::Zero(sum[part]);
    M::template Step<PARTS>(a_tile, b_tile, wm, wn, part, lane, sum[part]);
  }
#pragma unroll
  for (int part = 1; part < PARTS; ++part) M::Add(sum[0], sum[part]);
  M::Add(acc, sum[0]);
}

// The K loop over steps [s, s1): ta / tb are operand tiles with Load<guard>(registers, step, k, tid) and Store(LDS, ...);
// steps below full_steps need no guard.  `lds` holds two stages.
// PARTS > 0 (one K group): acc is a chain of steps and not of products.
template <typename T, bool A_KC, bool B_KC, int BM, int BN, int KG, int PARTS = 0, typename TA, typename TB>
__device__ __forceinline__ void KLoop(char* lds, TA& ta, TB& tb, int s, int s1, int full_steps, int k_total, int tid,
                                      typename Mma<T, A_KC, B_KC, BM, BN>::acc_t& acc) {
  constexpr int STAGE   = (BM + BN) * 128;
  constexpr int THREADS = 256 * KG;
  typedef Mma<T, A_KC, B_KC, BM, BN> M;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
  // A ring of PF steps in registers: the loads of step s + PF go out while step s is multiplied, PF - 1 steps of MFMAs
  // ahead of their use.  A small tile's step is shorter than a trip to memory.
  // (Two slots do not fit the registers of a 128x128 tile on four wavefronts beside a second block on the CU.)
  constexpr int PF = BM == 128 && KG == 1 ? 1 : 2;
  u32x4 ra[PF][BM * 8 / THREADS], rb[PF][BN * 8 / THREADS];
  auto load = [&](int step, int slot, bool whole) {
    if (whole) {
      ta.template Load<false>(ra[slot], step, k_total, tid);
      tb.template Load<false>(rb[slot], step, k_total, tid);
    } else {
      ta.template Load<true>(ra[slot], step, k_total, tid);
      tb.template Load<true>(rb[slot], step, k_total, tid);
    }
  };
  auto store = [&](int slot, char* stage) {
    ta.Store(stage, ra[slot], tid);
    tb.Store(stage + BM * 128, rb[slot], tid);
  };

  M::Zero(acc);
#pragma unroll
  for (int u = 0; u < PF; ++u)
    if (s + u < s1) load(s + u, u, s + u < full_steps);
  store(0, lds);
  __syncthreads();
  // pairs of steps (the LDS stage is a constant) that both have an unguarded step to request: no branches, so that the
  // compiler can count the loads in flight where it waits for one slot
  const int main1 = min(s1, full_steps) - PF;
  for (; s + 2 <= main1; s += 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      char* cur = lds + (u & 1) * STAGE;
      load(s + u + PF, u % PF, true);
      if constexpr (PARTS == 0) {
        M::template Step<KG>(cur, cur + BM * 128, wm, wn, kg, lane, acc);
      } else {
        InParts<M, PARTS>(cur, cur + BM * 128, wm, wn, lane, acc);
      }
      store((u + 1) % PF, lds + ((u + 1) & 1) * STAGE);
      __syncthreads();
    }
  }
  for (; s < s1; s += 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (s + u >= s1) break;
      char* cur = lds + (u & 1) * STAGE;
      if (s + u + PF < s1) load(s + u + PF, u % PF, s + u + PF < full_steps);
      if constexpr (PARTS == 0) {
        M::template Step<KG>(cur, cur + BM * 128, wm, wn, kg, lane, acc);
      } else {
        InParts<M, PARTS>(cur, cur + BM * 128, wm, wn, lane, acc);
      }
      if (s + u + 1 < s1) store((u + 1) % PF, lds + ((u + 1) & 1) * STAGE);
      __syncthreads();
    }
  }
}

// The block's result tile through LDS as fp32, 64 rows at a time: f(row, first column, eight values) for every group of
// eight columns, relative to the tile.  The LDS of the two stages is reused (the loop's last barrier has passed).
template <typename T, bool A_KC, bool B_KC, int BM, int BN, int KG, typename F>
__device__ __forceinline__ void EachRowGroup(char* lds, const typename Mma<T, A_KC, B_KC, BM, BN>::acc_t& acc, int tid, F f) {
  constexpr int PASSES  = BM / 64;
  constexpr int THREADS = 256 * KG;
  constexpr int SLD     = BN + 4;          // row pitch (floats): row groups of 4 land 16 banks apart
  constexpr int CPR     = BN / 8;          // eight-column groups per row
  constexpr int ROWS    = THREADS / CPR;   // rows per sweep
  static_assert(64 * SLD * 4 <= 2 * (BM + BN) * 128, "the staging tile fits the stages");
  typedef Mma<T, A_KC, B_KC, BM, BN> M;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
  float* st = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int pass = 0; pass < PASSES; ++pass) {
    if (pass > 0) __syncthreads();
    float* at = st + (PASSES == 1 ? wm * (BM / 2) * SLD : 0) + wn * (BN / 2);
#pragma unroll
    for (int g = 0; g < KG; ++g) {
      if (kg == g && (PASSES == 1 || wm == pass))
        M::Each(acc, lane, [&](int row, int col, float v) { at[row * SLD + col] = g == 0 ? v : at[row * SLD + col] + v; });
      __syncthreads();
    }
#pragma unroll 1
    for (int row = tid / CPR; row < 64; row += ROWS) {
      float v[8];
      const float* from = &st[row * SLD + (tid % CPR) * 8];
      *reinterpret_cast<f32x4*>(&v[0]) = *reinterpret_cast<const f32x4*>(from);
      *reinterpret_cast<f32x4*>(&v[4]) = *reinterpret_cast<const f32x4*>(from + 4);
      f(pass * 64 + row, (tid % CPR) * 8, v);
    }
  }
}

}  // namespace flex
}  // namespace cinn_hip_kernels
