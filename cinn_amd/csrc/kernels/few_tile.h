// Device code shared by the kernels of few output tiles (conv_few_mfma.hip, gemm_rows.hip): the wavefronts of a block split K among
// themselves, each has a ring of K steps of its own in LDS, filled by direct global -> LDS loads, waits for nobody and meets the
// others once, at the end.  A K step is 128 bytes of every row; a fragment is 16 rows.
//
// What a CU pulls in depends on the order of a load's lanes: sixteen-byte pieces of one 128-byte line in eight neighbouring lanes
// arrive at 125 GB/s per CU (operands in L2), the same bytes in the order of an MFMA fragment (sixteen rows in neighbouring
// lanes) at 37 GB/s.  So a load brings 8 rows of 128 bytes, eight lanes to a row, and fragments are read from LDS.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

namespace cinn_hip_kernels {
namespace few {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kStepBytes = 128;  // of a row, per K step

// 16 bytes of a row of each operand, in each of four lane groups: one 16x16x32 product, or four of 16x16x4.  The result has
// the rows of w as its rows: a lane ends up with four consecutive ones (4 (lane / 16) ..) of row lane % 16 of x.
template <typename T>
__device__ __forceinline__ f32x4 Multiply(u32x4 w, u32x4 x, f32x4 acc) {
  if constexpr (std::is_same<T, float>::value) {
    const f32x4 a = __builtin_bit_cast(f32x4, w), b = __builtin_bit_cast(f32x4, x);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc, 0, 0, 0);
    return acc;
  } else if constexpr (std::is_same<T, _Float16>::value) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, x), acc, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), acc, 0, 0, 0);
  }
}

// Place of 16-byte chunk c in row r of a fragment in LDS, and the chunk at a place.  A 16-byte read serves lanes 8 p .. 8 p + 7 with
// 32 + 8 p .. 32 + 8 p + 7, rows of one half with chunks that differ in bit 1: exchanged with bit 0 and varied by the row, the
// sixteen lie in sixteen groups of banks.
__device__ __forceinline__ int Swap01(int c) { return (c & 4) | ((c & 1) << 1) | ((c >> 1) & 1); }
__device__ __forceinline__ int PlaceOf(int c, int r) { return Swap01(c) ^ (r & 7) ^ (r >> 3); }
__device__ __forceinline__ int ChunkAt(int place, int r) { return Swap01(place ^ (r & 7) ^ (r >> 3)); }

// Direct global -> LDS loads of 16 bytes per lane, written at LDS address `to` + 16 * lane.  Inline assembly: loads that the
// compiler tracks are waited for before any LDS read.
__device__ __forceinline__ void CopyAt(unsigned to, const void* from) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(to), "v"(from) : "memory");
}
__device__ __forceinline__ void CopyAt(unsigned to, const void* base, unsigned offset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(to), "v"(offset), "s"(base) : "memory");
}
// at most N of the wavefront's loads in flight
template <int N>
__device__ __forceinline__ void WaitLoads() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ __forceinline__ void WaitLdsReads() { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); }

// The ring of a wavefront: SLOTS K steps of TM fragments of x (unless these lie elsewhere) and TN of w.
template <typename T, int TM, int TN, int SLOTS = 2, bool WITH_X = true>
struct Ring {
  static constexpr int FRAG  = 16 * kStepBytes;
  static constexpr int XS    = WITH_X ? TM : 0;
  static constexpr int SLOT  = (XS + TN) * FRAG;
  static constexpr int BYTES = SLOTS * SLOT;
  static constexpr int LOADS = 2 * (TM + TN);  // of a step
  char* at;
  unsigned address;  // the same for the loads
  int offset[2];     // of the lane's chunk of either half of a step in a fragment
  u32x4 xs[TM][2], ws[TN][2];
  f32x4 acc[TM][TN];

  __device__ __forceinline__ Ring(char* lds, int wave, int lane) : at(lds + wave * BYTES) {
    address = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) char*)at);
#pragma unroll
    for (int half = 0; half < 2; ++half) offset[half] = (lane & 15) * kStepBytes + (PlaceOf(half * 4 + (lane >> 4), lane & 15) << 4);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  // where load i of a step's rows of x (8 each), or load j of its rows of w, goes
  __device__ __forceinline__ unsigned X(int slot, int i) const { return address + slot * SLOT + i * (FRAG / 2); }
  __device__ __forceinline__ unsigned W(int slot, int j) const { return address + slot * SLOT + (2 * XS + j) * (FRAG / 2); }
  __device__ __forceinline__ void Read(int slot) {
    const char* from = at + slot * SLOT;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int j = 0; j < TN; ++j) ws[j][half] = *reinterpret_cast<const u32x4*>(from + (XS + j) * FRAG + offset[half]);
#pragma unroll
      for (int i = 0; i < XS; ++i) xs[i][half] = *reinterpret_cast<const u32x4*>(from + i * FRAG + offset[half]);
    }
  }
  __device__ __forceinline__ void Mma() {
    // fp32: the products of a step in a chain of their own, so that acc is a chain of steps and not of products.  (The tiled kernels
    // split K over more blocks than there are wavefronts here.  Relative error against float64 over theirs, 35 convolutions and 40
    // products: 0.83 and 0.79 in the geometric mean and up to 1.6 as one chain, 0.48 and 0.64 so and none above (a product of one
    // step is the same chain there: 0.98 to 1.01); as two chains a step 0.42 and 0.54.  Time 1.01 to 1.02 of one chain's, two chains 1.04.)
    if constexpr (sizeof(T) == 4) {
      f32x4 sum[TM][TN];
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            sum[i][j] = Multiply<T>(ws[j][half], xs[i][half], half == 0 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : sum[i][j]);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += sum[i][j];
      return;
    }
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = Multiply<T>(ws[j][half], xs[i][half], acc[i][j]);
  }
  // all of the wavefront's `steps` K steps, two in flight; request(slot) issues the LOADS loads of the next one
  template <typename F>
  __device__ __forceinline__ void Run(int steps, F request) {
    static_assert(WITH_X && SLOTS == 2, "the waits count the loads of one step");
    if (steps < 2) {
      if (steps == 1) {
        request(0);
        WaitLoads<0>();
        Read(0);
        Mma();
      }
      return;
    }
    request(0);
    request(1);
    for (; steps >= 4; steps -= 2) {
#pragma unroll
      for (int slot = 0; slot < 2; ++slot) {
        WaitLoads<LOADS>();
        Read(slot);
        WaitLdsReads();  // the slot is free
        request(slot);
        Mma();
      }
    }
    const int odd = steps - 2;  // one more step to request
    if (odd) {
      WaitLoads<LOADS>();
      Read(0);
      WaitLdsReads();
      request(0);
      Mma();
    }
    WaitLoads<LOADS>();
    Read(odd);
    Mma();
    WaitLoads<0>();
    Read(1 - odd);
    Mma();
  }
  // The parts meet in LDS, every wavefront's where its ring was.  f(n, i, j, sum) for the wavefront's n-th fragment to finish,
  // fragment (i, j) of the tile: the lane's four consecutive columns of one row.
  template <int NW, typename F>
  __device__ __forceinline__ void Meet(const char* lds, int wave, int lane, F f) {
    static_assert(TM * TN * 1024 <= BYTES, "the parts fit the rings");
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) *reinterpret_cast<f32x4*>(at + (i * TN + j) * 1024 + lane * 16) = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int n = 0; n < (TM * TN + NW - 1) / NW; ++n) {
      const int frag = wave + n * NW;
      if (frag >= TM * TN) continue;
      f32x4 sum = *reinterpret_cast<const f32x4*>(lds + frag * 1024 + lane * 16);
#pragma unroll
      for (int k = 1; k < NW; ++k) sum += *reinterpret_cast<const f32x4*>(lds + k * BYTES + frag * 1024 + lane * 16);
      f(n, frag / TN, frag % TN, sum);
    }
  }
};

// Tile (of a contiguous run of them for every XCD, which consecutive block ids visit in turn); `rows_outer`: neighbours share
// the rows of x (or of w).
__device__ __forceinline__ void TileOf(int bid, int tiles_m, int tiles_n, bool rows_outer, int* tm, int* tn) {
  const int tiles = tiles_m * tiles_n, q = tiles >> 3, rest = tiles & 7, xcd = bid & 7;
  const int id = xcd * q + min(xcd, rest) + (bid >> 3);
  *tm = rows_outer ? id / tiles_n : id % tiles_m;
  *tn = rows_outer ? id % tiles_n : id / tiles_m;
}

// A tile's launch, in us: a block's start and end, what its CU pulls in and multiplies, rounds of blocks beyond
// those that a CU holds.  The coefficients are fitted and not rates (147 bytes per ns, where a CU was seen to pull in 110 to 130, since part
// of that lies under the constant), to 330 layers of 1 to 32 images (0.14 in the logarithm, 2% from the best tile on average).
inline double Estimate(int rows, int cols, int steps, bool fp32, int tm, int tn, int nw) {
  const double blocks   = (double)((rows + 16 * tm - 1) / (16 * tm)) * ((cols + 16 * tn - 1) / (16 * tn)), per_cu = std::ceil(blocks / 256);
  const int resident    = std::min(160 / (nw * 2 * (tm + tn) * 2), 8);
  const double pulled   = per_cu * (tm + tn) * 2.048 * steps / 147;
  const double multiply = per_cu * steps * tm * tn * (fp32 ? 8 * 32 : 2 * 16) / 4 / 1938.0;
  return 3.0 + std::max(pulled, multiply) + 0.43 * std::min(pulled, multiply) + 1.15 * (std::ceil(per_cu / resident) - 1) + 0.043 * steps / nw;
}

}  // namespace few
}  // namespace cinn_hip_kernels
