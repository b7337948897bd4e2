// Register-staged MFMA matrix product for gfx950: any extents, any operand layout, any alignment, fp16 / bf16 / fp32.
//
//   C[m][n] = epilogue( sum_k A[m][k] B[k][n] ),  A stored [m][k] or [k][m], B stored [n][k] or [k][n]
//
// The direct-to-LDS kernels of gemm_mfma.hip need whole, aligned 16-byte chunks and a K-contiguous A.  Everything else
// comes here: transposed A (the weight gradient of a linear layer), extents that are no multiple of anything, many
// small batch entries.  What it does instead:
//   * an operand keeps its own order on the way into LDS: a K-contiguous one as [row][128 bytes of k], the other as
//     [k][rows].  Fragments of the latter are read with ds_read_b64_tr_b16 (16-bit) or as single floats, so nothing is
//     transposed in registers or in memory beforehand;
//   * chunks travel global -> registers -> LDS, one K step ahead: a global load takes any element-aligned address and a
//     chunk can be masked.  Chunks that reach beyond K, or beyond the end of the operand's last row, only occur in the
//     last step or two of a product; those run a guarded loader, all others an unguarded one;
//   * rows beyond M / N repeat the last one; what they produce is not stored;
//   * grids too small for the chip split K over blockIdx.z, and a second kernel adds the fp32 planes.
// Measured before (transposing copies in front of a convolution kernel, one launch per batch entry, or scalar FMAs
// where K was no multiple of a chunk) and here, us: fp16 A^T B 768 x 3072 x 4100 871 -> 39 (495 TFLOP/s), [64] x 1 x 215
// x 48 262 -> 4.0, 1000^3 15.3 -> 10.4; bf16 [2] x 2336 x 3250 x 153 120 -> 25, 512 x 512 x 4096 26 -> 14; fp32 1000^3
// 36 -> 24 (84 TFLOP/s), A^T B 768 x 3072 x 4100 218 -> 171 (113 TFLOP/s).  A step of a 64x64 tile is bound by the trip of its chunks to LDS
// (0.42 us for a block alone), of a 128x128 tile by the register staging around its MFMAs (0.6 us for 0.2 of MFMA).
#include "kernels/gemm_flex.h"

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <type_traits>

#include "runtime/hip_check.h"
#include "runtime/scratch.h"

namespace cinn_hip_kernels {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

struct FlexParams {
  const void* a;
  const void* b;
  void* c;
  float* partials;  // fp32 planes [split][batch][m][n] of a split reduction, or null
  int m, n, k;
  int64_t lda, ldb;
  int64_t stride_a, stride_b, stride_c;
  int tiles_m, tiles_n;
  int steps;            // K steps of 128 bytes
  int steps_per_split;
  int full_steps;       // the first full_steps steps read nothing beyond K or beyond an operand's end
  const float* scale;
  const float* shift;
  const void* residual;
  float alpha, residual_scale;
  int relu;
};

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

// `residual` is 0 where there is none
__device__ __forceinline__ float Finish(float v, float scale, float shift, float residual_scale, float residual, int relu) {
  v = __builtin_fmaf(residual_scale, residual, __builtin_fmaf(v, scale, shift));
  return relu ? fmaxf(v, 0.0f) : v;
}

// KG groups of four wavefronts (2 x 2 over the tile) share the block's tiles and take a K step's slices in turn; their
// sums meet in the epilogue.  Two groups where the grid puts at most two blocks on a CU: with one wavefront per SIMD
// nobody multiplies while it waits for LDS or writes the next step's chunks.
template <typename T, bool A_KC, bool B_KC, int BM, int BN, int KG>
__global__ void __launch_bounds__(256 * KG)
flex_gemm_kernel(FlexParams p) {
  constexpr int THREADS = 256 * KG;
  constexpr int STAGE = (BM + BN) * 128;
  constexpr int SLD   = BN + 4;  // row pitch (floats) of the epilogue's staging tile: row groups of 4 land 16 banks apart
  constexpr int LDS   = 2 * STAGE > 64 * SLD * 4 ? 2 * STAGE : 64 * SLD * 4;
  __shared__ __attribute__((aligned(256))) char lds[LDS];
  const int tid  = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
  int tm, tn;
  TileOf(blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN;

  Tile<T, A_KC, BM, THREADS> ta;
  Tile<T, B_KC, BN, THREADS> tb;
  ta.Init(static_cast<const T*>(p.a) + blockIdx.y * p.stride_a, p.lda, m0, p.m, p.k, tid);
  tb.Init(static_cast<const T*>(p.b) + blockIdx.y * p.stride_b, p.ldb, n0, p.n, p.k, tid);
  // A ring of PF steps in registers: the loads of step s + PF go out while step s is multiplied, PF - 1 steps of MFMAs
  // ahead of their use.  A small tile's step is shorter than a trip to memory.
  // (Two slots do not fit the registers of a 128x128 tile on four wavefronts beside a second block on the CU.)
  constexpr int PF = BM == 128 && KG == 1 ? 1 : 2;
  u32x4 ra[PF][BM * 8 / THREADS], rb[PF][BN * 8 / THREADS];
  auto load = [&](int step, int slot, bool whole) {
    if (whole) {
      ta.template Load<false>(ra[slot], step, p.k, tid);
      tb.template Load<false>(rb[slot], step, p.k, tid);
    } else {
      ta.template Load<true>(ra[slot], step, p.k, tid);
      tb.template Load<true>(rb[slot], step, p.k, tid);
    }
  };
  auto store = [&](int slot, char* stage) {
    ta.Store(stage, ra[slot], tid);
    tb.Store(stage + BM * 128, rb[slot], tid);
  };

  typedef Mma<T, A_KC, B_KC, BM, BN> M;
  typename M::acc_t acc;
  M::Zero(acc);
  int s        = blockIdx.z * p.steps_per_split;
  const int s1 = min(s + p.steps_per_split, p.steps);
#pragma unroll
  for (int u = 0; u < PF; ++u)
    if (s + u < s1) load(s + u, u, s + u < p.full_steps);
  store(0, lds);
  __syncthreads();
  // pairs of steps (the LDS stage is a constant) that both have an unguarded step to request: no branches, so that the
  // compiler can count the loads in flight where it waits for one slot
  const int main1 = min(s1, p.full_steps) - PF;
  for (; s + 2 <= main1; s += 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      char* cur = lds + (u & 1) * STAGE;
      load(s + u + PF, u % PF, true);
      M::template Step<KG>(cur, cur + BM * 128, wm, wn, kg, lane, acc);
      store((u + 1) % PF, lds + ((u + 1) & 1) * STAGE);
      __syncthreads();
    }
  }
  for (; s < s1; s += 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (s + u >= s1) break;
      char* cur = lds + (u & 1) * STAGE;
      if (s + u + PF < s1) load(s + u + PF, u % PF, s + u + PF < p.full_steps);
      M::template Step<KG>(cur, cur + BM * 128, wm, wn, kg, lane, acc);
      if (s + u + 1 < s1) store((u + 1) % PF, lds + ((u + 1) & 1) * STAGE);
      __syncthreads();
    }
  }

  // Epilogue: 64 rows at a time through LDS as fp32, then eight columns of one row per thread.
  constexpr int PASSES = BM / 64;
  constexpr int CPR    = BN / 8;          // eight-column groups per row
  constexpr int ROWS   = THREADS / CPR;   // rows per sweep
  float* st      = reinterpret_cast<float*>(lds);
  const int col0 = n0 + (tid % CPR) * 8;
  const int cols = min(p.n - col0, 8);
  float sc[8], sh[8];
  if (!p.partials) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int col = min(col0 + e, p.n - 1);
      sc[e] = p.scale ? p.scale[col] : p.alpha;
      sh[e] = p.shift ? p.shift[col] : 0.0f;
    }
  }
  T* c              = static_cast<T*>(p.c) + blockIdx.y * p.stride_c;
  const T* residual = p.residual ? static_cast<const T*>(p.residual) + blockIdx.y * p.stride_c : nullptr;
  float* plane      = p.partials + ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * p.m * p.n;
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
    for (int row = tid / CPR; row < 64; row += ROWS) {
      const int m = m0 + pass * 64 + row;
      if (m >= p.m || cols <= 0) break;
      float v[8];
      *reinterpret_cast<f32x4*>(&v[0]) = *reinterpret_cast<const f32x4*>(&st[row * SLD + (tid % CPR) * 8]);
      *reinterpret_cast<f32x4*>(&v[4]) = *reinterpret_cast<const f32x4*>(&st[row * SLD + (tid % CPR) * 8 + 4]);
      const int64_t at = (int64_t)m * p.n + col0;
      if (p.partials) {
        if (cols == 8) {
          __builtin_memcpy(plane + at, v, 32);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (e < cols) plane[at + e] = v[e];
        }
        continue;
      }
      if (cols == 8) {
        typedef T vec8 __attribute__((ext_vector_type(8)));
        vec8 out, res = {0, 0, 0, 0, 0, 0, 0, 0};
        if (residual) __builtin_memcpy(&res, residual + at, 8 * sizeof(T));
#pragma unroll
        for (int e = 0; e < 8; ++e) out[e] = (T)Finish(v[e], sc[e], sh[e], p.residual_scale, (float)res[e], p.relu);
        __builtin_memcpy(c + at, &out, 8 * sizeof(T));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (e < cols)
            c[at + e] = (T)Finish(v[e], sc[e], sh[e], p.residual_scale, residual ? (float)residual[at + e] : 0.0f, p.relu);
      }
    }
  }
}

// Adds the planes of a split reduction and applies the epilogue: one thread per V consecutive elements of a plane row
// (V divides n), planes in ascending order.
template <typename T, int V>
__global__ void __launch_bounds__(256)
flex_reduce_kernel(FlexParams p, int splits, int64_t plane) {
  const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (at >= plane) return;
  float v[V];
  __builtin_memcpy(v, p.partials + at, V * 4);
#pragma unroll 4
  for (int s = 1; s < splits; ++s) {
    float w[V];
    __builtin_memcpy(w, p.partials + s * plane + at, V * 4);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] += w[e];
  }
  // batch entries of a split product are dense: an element's place in a plane is its place in C
  const int col = (int)(at % p.n);
  T out[V], res[V];
#pragma unroll
  for (int e = 0; e < V; ++e) res[e] = (T)0.0f;
  if (p.residual) __builtin_memcpy(res, static_cast<const T*>(p.residual) + at, V * sizeof(T));
#pragma unroll
  for (int e = 0; e < V; ++e)
    out[e] = (T)Finish(v[e], p.scale ? p.scale[col + e] : p.alpha, p.shift ? p.shift[col + e] : 0.0f, p.residual_scale,
                       (float)res[e], p.relu);
  __builtin_memcpy(static_cast<T*>(p.c) + at, out, V * sizeof(T));
}

// K steps that neither loader has to guard
template <typename T>
int FullSteps(bool kc, int64_t ld, int rows, int k) {
  constexpr int E = 16 / (int)sizeof(T), KS = 8 * E;
  if (kc) return k / KS;
  // the last chunk of a k row reaches up to E - 1 elements beyond the row, which is fine while that is still inside
  // the operand
  const int64_t room = (int64_t)(k - 1) * ld + rows - (int64_t)(rows + E - 1) / E * E;
  return room < 0 ? 0 : (int)((std::min<int64_t>(room / ld, k - 1) + 1) / KS);
}

struct Plan {
  int tile, kg, splits;
};

// Block tile and K split with the smallest estimated time.  The estimate (us) adds, per CU, the K steps of the blocks
// it gets, and what a split writes and reads back.  A block alone on its CU takes `alone` per step, blocks that share
// one take `shared` each, at most `resident` at a time; measured on a product of 768 x 3072 x 4100 (A and B [k][rows]),
// 2048^3, 1000^3 and 512 x 512 x 4096 with every tile and 1, 4 and 8 splits, which the estimate ranks as measured:
// 16-bit 768 x 3072 x 4100 39 us on 128x128 tiles of two groups, 46 on 64x64 tiles, 2048^3 26 / 33, 1000^3 17 / 10;
// [2] x 2336 x 3250 x 153 25 us on 128x128 tiles of one group (two blocks per CU cover each other's epilogue) against
// 40 with two; fp32 768 x 3072 x 4100 262 us on 128x128 tiles, 205 on 64x64 and 170 with K split four ways: a step is
// bound by the matrix pipe there, and small tiles spread evenly.
Plan ChoosePlan(const FlexGemm& g, int steps) {
  struct Shape {
    int tile, kg, resident;
    double alone, shared;
  };
  static const Shape k16[] = {{64, 1, 4, 0.42, 0.21}, {128, 1, 2, 0.87, 0.55}, {128, 2, 1, 0.62, 0.62}};
  static const Shape k32[] = {{64, 1, 4, 0.62, 0.50}};
  const bool fp32    = g.type == FlexType::kF32;
  const Shape* shape = fp32 ? k32 : k16;
  const int shapes   = fp32 ? 1 : 3;
  const double plane = (double)g.batch * g.m * g.n;
  Plan best{64, 1, 1};
  double least = 1e30;
  for (int i = 0; i < shapes; ++i) {
    const Shape& t = shape[i];
    const double tiles = (double)((g.m + t.tile - 1) / t.tile) * ((g.n + t.tile - 1) / t.tile) * g.batch;
    for (int splits = 1; splits <= 16 && (splits == 1 || steps / splits >= 4); ++splits) {
      const int per_cu    = (int)((tiles * splits + 255) / 256);
      const int rounds    = per_cu / t.resident, rest = per_cu % t.resident;
      const double round  = std::max(t.alone, t.shared * t.resident);
      const double a_step = rounds * round + (rest ? std::max(t.alone, t.shared * rest) : 0.0);
      // a block's start and epilogue: about two steps' worth
      double us = a_step * ((steps + splits - 1) / splits + 2);
      if (splits > 1) us += 4.0 + splits * plane * 8.0 / 4e6;
      if (us < least) least = us, best = {t.tile, t.kg, splits};
    }
  }
  return best;
}

template <typename T, bool A_KC, bool B_KC>
void LaunchTiles(const Plan& plan, dim3 grid, const FlexParams& p, hipStream_t stream) {
  if (plan.tile == 64) {
    hipLaunchKernelGGL((flex_gemm_kernel<T, A_KC, B_KC, 64, 64, 1>), grid, dim3(256), 0, stream, p);
    return;
  }
  if constexpr (sizeof(T) == 2) {
    if (plan.kg == 2) {
      hipLaunchKernelGGL((flex_gemm_kernel<T, A_KC, B_KC, 128, 128, 2>), grid, dim3(512), 0, stream, p);
    } else {
      hipLaunchKernelGGL((flex_gemm_kernel<T, A_KC, B_KC, 128, 128, 1>), grid, dim3(256), 0, stream, p);
    }
  }
}

template <typename T>
void Launch(const FlexGemm& g, hipStream_t stream) {
  constexpr int KS = 128 / (int)sizeof(T);
  FlexParams p;
  p.a = g.a, p.b = g.b, p.c = g.c;
  p.m = g.m, p.n = g.n, p.k = g.k;
  p.lda = g.lda, p.ldb = g.ldb;
  p.stride_a = g.stride_a, p.stride_b = g.stride_b, p.stride_c = g.stride_c;
  p.steps      = (g.k + KS - 1) / KS;
  p.full_steps = std::min(FullSteps<T>(g.a_kc, g.lda, g.m, g.k), FullSteps<T>(g.b_kc, g.ldb, g.n, g.k));
  p.scale = g.scale, p.shift = g.shift, p.residual = g.residual;
  p.alpha = g.alpha, p.residual_scale = g.residual_scale, p.relu = g.relu ? 1 : 0;
  Plan plan         = ChoosePlan(g, p.steps);
  p.steps_per_split = (p.steps + plan.splits - 1) / plan.splits;
  plan.splits       = (p.steps + p.steps_per_split - 1) / p.steps_per_split;
  p.tiles_m         = (g.m + plan.tile - 1) / plan.tile;
  p.tiles_n         = (g.n + plan.tile - 1) / plan.tile;
  const int64_t plane = (int64_t)g.batch * g.m * g.n;
  p.partials = plan.splits > 1 ? static_cast<float*>(Scratch(ScratchKind::kSplitK, (size_t)plan.splits * plane * sizeof(float), stream))
                               : nullptr;
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), g.batch, plan.splits);
  if (g.a_kc && g.b_kc) LaunchTiles<T, true, true>(plan, grid, p, stream);
  if (g.a_kc && !g.b_kc) LaunchTiles<T, true, false>(plan, grid, p, stream);
  if (!g.a_kc && g.b_kc) LaunchTiles<T, false, true>(plan, grid, p, stream);
  if (!g.a_kc && !g.b_kc) LaunchTiles<T, false, false>(plan, grid, p, stream);
  if (plan.splits > 1) {
    if (g.n % 4 == 0) {
      hipLaunchKernelGGL((flex_reduce_kernel<T, 4>), dim3((unsigned)((plane / 4 + 255) / 256)), dim3(256), 0, stream, p,
                         plan.splits, plane);
    } else {
      hipLaunchKernelGGL((flex_reduce_kernel<T, 1>), dim3((unsigned)((plane + 255) / 256)), dim3(256), 0, stream, p, plan.splits,
                         plane);
    }
  }
  CINN_HIP_CALL(hipGetLastError());
}

}  // namespace

bool TryFlexGemm(const FlexGemm& g, hipStream_t stream) {
  const int elem = g.type == FlexType::kF32 ? 4 : 2;
  // a thread's chunk is a 32-bit byte offset from the tile's first element: 128 rows, or 64 k rows, of the operand
  const int64_t limit = ((int64_t)1 << 31) / (128 * elem);
  if (g.lda >= limit || g.ldb >= limit) return false;
  const int64_t tiles = (int64_t)((g.m + 63) / 64) * ((g.n + 63) / 64);
  if (tiles >= INT_MAX / 8 || g.batch > 65535) return false;
  switch (g.type) {
    case FlexType::kF16: Launch<_Float16>(g, stream); break;
    case FlexType::kBF16: Launch<__bf16>(g, stream); break;
    case FlexType::kF32: Launch<float>(g, stream); break;
  }
  return true;
}

}  // namespace cinn_hip_kernels
