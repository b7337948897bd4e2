// Products of few rows for gfx950 (M <= 64: a classifier at inference batch sizes, a decoding step), fp16 / bf16:
//   C [M][N] = act( norm(A) [M][K] . B [N][K]^T * scale + shift + residual )
//
// Bound by one pass over B.  The tiled kernels give such a product M-tiles that are mostly padding and a handful of blocks;
// here small tiles give most CUs a block and its wavefronts split K.
//   * gemm_rows_ring_kernel: whole K steps of 64 in aligned rows, operands through rings in LDS in whole lines (few_tile.h: a CU
//     pulls in three times as much that way);
//   * gemm_rows_kernel: any other K of 32-deep blocks, operands at any address of their type, and some single rows (OneRow).  A block owns 16 output columns of
//     MT row tiles, its eight wavefronts split K, fragments come straight from global memory, 2 U k-blocks of loads in flight.
// us, the latter | the former, fp16: 8 x 768 -> 768 4.1 | 3.3, 8 x 3072 -> 768 7.2 | 4.7, 64 x 1280 -> 5120 24.7 | 6.4, 16 x 4096 -> 4096 with gelu 10.4 |
// 6.1; norm inside 8 x 768 -> 3072 5.4 | 4.1, with gelu 6.0 | 4.6.
//
// At these sizes a launch costs as much as the product (an empty kernel 3.3 us from launch to launch, 8 x 768 -> 768 5 us),
// so what surrounds the product in a decoding step is part of it:
//   * NORM: the layer norm of A's rows.  Every block has the rows' elements in registers anyway; sums of x and x x over a
//     lane's k, its row's other lanes and wavefronts (through LDS) give mean and variance, and the fragments are normalised
//     where they are.  One block barrier more;
//   * gelu, on the fp32 sum;
//   * several result tensors side by side (query, key and value of a token), each a contiguous matrix of its own.
// A block of one new token per sequence (8 sequences, hidden 768, 12 heads, 511 cached, fp16): nine launches in 46.0 us
// before, five in 28.8 here (35.9 with fragments straight from memory).
#include "kernels/gemm_rows.h"

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <type_traits>

#include "cinn_hip_runtime.h"
#include "kernels/few_tile.h"
#include "kernels/launch_count.h"
#include "runtime/hip_check.h"

namespace cinn_hip_kernels {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <typename T>
struct Half16;
template <>
struct Half16<__bf16> {
  typedef bf16x8 vec8;
  typedef bf16x8 loaded __attribute__((aligned(2)));  // 16 bytes at any element's address: the same load instruction
  static __device__ __forceinline__ f32x4 mfma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Half16<_Float16> {
  typedef f16x8 vec8;
  typedef f16x8 loaded __attribute__((aligned(2)));
  static __device__ __forceinline__ f32x4 mfma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

constexpr int NW = 8;  // wavefronts of a block
// k-blocks of a wavefront that a normalised row keeps in registers
constexpr int kNormBlocks = kRowProductMaxNormK / 32 / NW;

template <typename T, int MT, bool NORM, bool GELU>
__global__ void __launch_bounds__(64 * NW)
gemm_rows_kernel(RowProduct p) {
  typedef typename Half16<T>::vec8 vec8;
  typedef typename Half16<T>::loaded loaded;
  static_assert(!NORM || MT == 1, "rows are normalised by blocks of one row tile");
  __shared__ __attribute__((aligned(16))) float s_part[NW][MT][64][4];
  __shared__ float s_sum[NORM ? NW : 1][16][2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0   = blockIdx.x * 16;
  const int m0   = blockIdx.y * (MT * 16);  // first of this block's rows
  const int fr   = lane & 15;               // row of the fragment this lane reads (a row of A, a column of C for B)
  const int fk   = (lane >> 4) * 8;         // its 8 elements of a 32-deep k block
  // this wavefront's k-blocks: `mine` consecutive ones (neighbours share 128-byte lines), none when K is short
  const int blocks = p.k / 32, share = (blocks + NW - 1) / NW;
  const int first = min(wave * share, blocks - 1);
  const int mine  = min(share, blocks - wave * share);
  const T* bp     = static_cast<const T*>(p.b) + (int64_t)min(n0 + fr, p.n - 1) * p.k + first * 32 + fk;
  const T* ap[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) ap[t] = static_cast<const T*>(p.a) + (int64_t)min(m0 + t * 16 + fr, p.m - 1) * p.k + first * 32 + fk;
  // offset of block `i`; beyond the share the last one again (not multiplied)
  auto k_of = [&](int i) { return max(min(i, mine - 1), 0) * 32; };
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (NORM) {
    vec8 af[kNormBlocks], bf[kNormBlocks], g[kNormBlocks], be[kNormBlocks];
#pragma unroll
    for (int i = 0; i < kNormBlocks; ++i) af[i] = *reinterpret_cast<const loaded*>(ap[0] + k_of(i));
#pragma unroll
    for (int i = 0; i < kNormBlocks; ++i) {
      bf[i] = *reinterpret_cast<const loaded*>(bp + k_of(i));
      g[i]  = *reinterpret_cast<const loaded*>(static_cast<const T*>(p.gamma) + first * 32 + fk + k_of(i));
      be[i] = *reinterpret_cast<const loaded*>(static_cast<const T*>(p.beta) + first * 32 + fk + k_of(i));
    }
    float s = 0.0f, q = 0.0f;
#pragma unroll
    for (int i = 0; i < kNormBlocks; ++i)
      if (i < mine) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float x = (float)af[i][e];
          s += x;
          q = __builtin_fmaf(x, x, q);
        }
      }
    s += __shfl_xor(s, 16), q += __shfl_xor(q, 16);
    s += __shfl_xor(s, 32), q += __shfl_xor(q, 32);
    if (lane < 16) s_sum[wave][lane][0] = s, s_sum[wave][lane][1] = q;
    __syncthreads();
    s = q = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) s += s_sum[w][fr][0], q += s_sum[w][fr][1];
    const float mean = s / (float)p.k;
    const float var  = fmaxf(q / (float)p.k - mean * mean, 0.0f);
    const float inv  = 1.0f / sqrtf(var + p.epsilon);
#pragma unroll
    for (int i = 0; i < kNormBlocks; ++i)
      if (i < mine) {
        vec8 x;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (T)__builtin_fmaf(((float)af[i][e] - mean) * inv, (float)g[i][e], (float)be[i][e]);
        acc[0] = Half16<T>::mfma(x, bf[i], acc[0]);
      }
  } else {
    constexpr int U = 4;  // k-blocks per register set
    vec8 bf[2][U], af[2][U][MT];
    auto request = [&](int set, int i0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k_of(i0 + u);
        bf[set][u]  = *reinterpret_cast<const loaded*>(bp + k);
#pragma unroll
        for (int t = 0; t < MT; ++t) af[set][u][t] = *reinterpret_cast<const loaded*>(ap[t] + k);
      }
    };
    auto multiply = [&](int set, int i0) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (i0 + u < mine) {
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[t] = Half16<T>::mfma(af[set][u][t], bf[set][u], acc[t]);
        }
    };
    request(0, 0);
    for (int i = 0; i < mine; i += 2 * U) {
      if (i + U < mine) request(1, i + U);
      multiply(0, i);
      if (i + 2 * U < mine) request(0, i + 2 * U);
      multiply(1, i + U);
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) *reinterpret_cast<f32x4*>(&s_part[wave][t][lane][0]) = acc[t];
  __syncthreads();
  if (wave >= MT) return;
  // wavefront t: row tile t.  Lane = (column n0 + lane % 16, rows 16 t + 4 (lane / 16) .. + 3)
  f32x4 sum = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int w = 0; w < NW; ++w) sum += *reinterpret_cast<const f32x4*>(&s_part[w][wave][lane][0]);
  const int col = n0 + fr;
  if (col >= p.n) return;
  const float sc  = p.scale ? p.scale[col] : p.alpha;
  const float sh  = p.shift ? p.shift[col] : 0.0f;
  const int width = p.width;  // of a result tensor
  const int part  = (col >= width) + (col >= 2 * width);
  T* to           = static_cast<T*>(part == 0 ? p.c[0] : part == 1 ? p.c[1] : p.c[2]) + (col - part * width);
  const T* res    = static_cast<const T*>(p.residual);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = m0 + wave * 16 + 4 * (lane >> 4) + r;
    if (row >= p.m) continue;
    float v = __builtin_fmaf(sum[r], sc, sh);
    if (res) v = __builtin_fmaf(p.residual_scale, (float)res[(int64_t)row * p.n + col], v);
    asm volatile("" : "+v"(v));  // fp32 first, then one rounding to T: the same for every row
    if (p.relu) v = v > 0.0f ? v : 0.0f;
    if constexpr (GELU) v = v * __builtin_fmaf(0.5f, erff(v * 0.70710678f), 0.5f);
    to[(int64_t)row * width] = (T)v;
  }
}

// ---- whole, aligned K steps of 64: operands through rings in LDS (few_tile.h) ------------------------------------------
using few::u32x4;

// NORM: K steps of a wavefront that hold its share of a normalised row (0: no norm).  A's are requested at once and have LDS of
// their own; the rows' sums of x and x x run while B's are on their way, then fragments are normalised between LDS and the
// product.  B is requested at once too where a block has a CU to itself (TN = 1: 8 x 768 -> 3072 4.1 us, two steps at a time
// 4.5), two steps at a time where rounds of blocks want its LDS (1 x 1280 -> 9984 9.7 | 7.8).
template <typename T, int TM, int TN, int WAVES, int NORM>
__global__ void __launch_bounds__(64 * WAVES)
gemm_rows_ring_kernel(RowProduct p, int tiles_m, int tiles_n) {
  constexpr int SLOTS = NORM && TN == 1 ? std::max(NORM, 2) : 2;
  typedef few::Ring<T, TM, TN, SLOTS, NORM == 0> Ring;
  typedef typename Half16<T>::vec8 vec8;
  typedef T vec4 __attribute__((ext_vector_type(4)));
  static_assert(!NORM || TM == 1, "rows are normalised by blocks of one row tile");
  __shared__ __attribute__((aligned(1024))) char lds[WAVES * Ring::BYTES];
  __shared__ __attribute__((aligned(1024))) char rows[NORM ? WAVES * NORM * Ring::FRAG : 16];
  __shared__ float s_sum[NORM ? WAVES : 1][16][2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Ring ring(lds, wave, lane);
  int tm, tn;
  few::TileOf(blockIdx.x, tiles_m, tiles_n, false, &tm, &tn);
  const int m0 = tm * (16 * TM), n0 = tn * (16 * TN);
  const int row_bytes = p.k * 2, steps = p.k / 64;
  unsigned a_off[2 * TM], b_off[2 * TN];  // of the lane's chunks; rows beyond the last repeat it
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i)
    a_off[i] = (unsigned)min(m0 + 8 * i + (lane >> 3), p.m - 1) * (unsigned)row_bytes + (few::ChunkAt(lane & 7, 8 * (i & 1) + (lane >> 3)) << 4);
#pragma unroll
  for (int j = 0; j < 2 * TN; ++j)
    b_off[j] = (unsigned)min(n0 + 8 * j + (lane >> 3), p.n - 1) * (unsigned)row_bytes + (few::ChunkAt(lane & 7, 8 * (j & 1) + (lane >> 3)) << 4);
  // what the epilogue reads, see below
  constexpr int FINISH = (TM * TN + WAVES - 1) / WAVES;
  f32x4 sc[FINISH], sh[FINISH];
  vec4 res[FINISH];
#pragma unroll
  for (int f = 0; f < FINISH; ++f) {
    const int frag = wave + f * WAVES, row = m0 + 16 * (frag / TN) + (lane & 15), col = n0 + 16 * (frag % TN) + (lane >> 4) * 4;
    const bool mine = frag < TM * TN && row < p.m && col < p.n;
    sc[f]  = f32x4{p.alpha, p.alpha, p.alpha, p.alpha};
    sh[f]  = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    res[f] = vec4{(T)0.0f, (T)0.0f, (T)0.0f, (T)0.0f};
    if (mine && p.scale) sc[f] = *reinterpret_cast<const f32x4*>(p.scale + col);
    if (mine && p.shift) sh[f] = *reinterpret_cast<const f32x4*>(p.shift + col);
    if (mine && p.residual) res[f] = *reinterpret_cast<const vec4*>(static_cast<const T*>(p.residual) + (int64_t)row * p.n + col);
  }
  const int s0 = steps * wave / WAVES, mine = steps * (wave + 1) / WAVES - s0;
  const char* a = static_cast<const char*>(p.a) + (int64_t)s0 * few::kStepBytes;
  const char* b = static_cast<const char*>(p.b) + (int64_t)s0 * few::kStepBytes;
  if constexpr (NORM == 0) {
    ring.Run(mine, [&](int slot) {
#pragma unroll
      for (int j = 0; j < 2 * TN; ++j) few::CopyAt(ring.W(slot, j), b, b_off[j]);
#pragma unroll
      for (int i = 0; i < 2 * TM; ++i) few::CopyAt(ring.X(slot, i), a, a_off[i]);
      a += few::kStepBytes, b += few::kStepBytes;
    });
  } else {
    vec8 g[NORM][2], be[NORM][2];
#pragma unroll
    for (int d = 0; d < NORM; ++d)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int k  = (s0 + max(min(d, mine - 1), 0)) * 64 + half * 32 + (lane >> 4) * 8;
        g[d][half]  = *reinterpret_cast<const vec8*>(static_cast<const T*>(p.gamma) + k);
        be[d][half] = *reinterpret_cast<const vec8*>(static_cast<const T*>(p.beta) + k);
      }
    const char* my_rows     = rows + wave * NORM * Ring::FRAG;
    const unsigned rows_at = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) char*)my_rows);
#pragma unroll
    for (int d = 0; d < NORM; ++d)
      if (d < mine) {
#pragma unroll
        for (int i = 0; i < 2; ++i) few::CopyAt(rows_at + d * Ring::FRAG + i * (Ring::FRAG / 2), a + d * few::kStepBytes, a_off[i]);
      }
    auto request = [&](int d) {
#pragma unroll
      for (int j = 0; j < 2 * TN; ++j) few::CopyAt(ring.W(d % SLOTS, j), b + d * few::kStepBytes, b_off[j]);
    };
#pragma unroll
    for (int d = 0; d < NORM && d < SLOTS; ++d)
      if (d < mine) request(d);
    switch (min(mine, SLOTS)) {  // A is there, B may be on its way
      case 0: break;
      case 1: few::WaitLoads<2 * TN>(); break;
      case 2: few::WaitLoads<4 * TN>(); break;
      case 3: few::WaitLoads<6 * TN>(); break;
      case 4: few::WaitLoads<8 * TN>(); break;
      default: few::WaitLoads<10 * TN>(); break;
    }
    float s = 0.0f, q = 0.0f;
    vec8 x[NORM][2];
#pragma unroll
    for (int d = 0; d < NORM; ++d)
      if (d < mine) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          x[d][half] = *reinterpret_cast<const vec8*>(my_rows + d * Ring::FRAG + ring.offset[half]);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float v = (float)x[d][half][e];
            s += v;
            q = __builtin_fmaf(v, v, q);
          }
        }
      }
    s += __shfl_xor(s, 16), q += __shfl_xor(q, 16);
    s += __shfl_xor(s, 32), q += __shfl_xor(q, 32);
    if (lane < 16) s_sum[wave][lane][0] = s, s_sum[wave][lane][1] = q;
    __syncthreads();
    s = q = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) s += s_sum[w][lane & 15][0], q += s_sum[w][lane & 15][1];
    const float mean = s / (float)p.k;
    const float var  = fmaxf(q / (float)p.k - mean * mean, 0.0f);
    const float inv  = 1.0f / sqrtf(var + p.epsilon);
#pragma unroll
    for (int d = 0; d < NORM; ++d)
      if (d < mine) {
        if (SLOTS >= NORM) {
          if (d == 0) few::WaitLoads<0>();
        } else if (d + 1 < mine) {
          few::WaitLoads<2 * TN>();
        } else {
          few::WaitLoads<0>();
        }
        ring.Read(d % SLOTS);
        if (d + SLOTS < NORM && d + SLOTS < mine) {
          few::WaitLdsReads();  // the slot is free
          request(d + SLOTS);
        }
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          vec8 y;
#pragma unroll
          for (int e = 0; e < 8; ++e) y[e] = (T)__builtin_fmaf(((float)x[d][half][e] - mean) * inv, (float)g[d][half][e], (float)be[d][half][e]);
#pragma unroll
          for (int j = 0; j < TN; ++j) ring.acc[0][j] = few::Multiply<T>(ring.ws[j][half], __builtin_bit_cast(u32x4, y), ring.acc[0][j]);
        }
      }
  }
  ring.template Meet<WAVES>(lds, wave, lane, [&](int f, int i, int j, f32x4 sum) {
    const int row = m0 + 16 * i + (lane & 15), col = n0 + 16 * j + (lane >> 4) * 4;
    if (row >= p.m || col >= p.n) return;
    const int part = (col >= p.width) + (col >= 2 * p.width);
    T* to          = static_cast<T*>(part == 0 ? p.c[0] : part == 1 ? p.c[1] : p.c[2]) + (int64_t)row * p.width + (col - part * p.width);
    vec4 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = __builtin_fmaf(sum[e], sc[f][e], sh[f][e]);
      if (p.residual) v = __builtin_fmaf(p.residual_scale, (float)res[f][e], v);
      asm volatile("" : "+v"(v));  // fp32 first, then one rounding to T: the same for every row
      if (p.relu) v = v > 0.0f ? v : 0.0f;
      if (p.gelu) v = v * __builtin_fmaf(0.5f, erff(v * 0.70710678f), 0.5f);
      out[e] = (T)v;
    }
    *reinterpret_cast<vec4*>(to) = out;
  });
}

template <typename T, int TM, int TN, int WAVES, int NORM>
void LaunchRing(const RowProduct& p, hipStream_t stream) {
  const int tiles_m = (p.m + 16 * TM - 1) / (16 * TM), tiles_n = (p.n + 16 * TN - 1) / (16 * TN);
  hipLaunchKernelGGL((gemm_rows_ring_kernel<T, TM, TN, WAVES, NORM>), dim3((unsigned)(tiles_m * tiles_n)), dim3(64 * WAVES), 0, stream, p, tiles_m,
                     tiles_n);
}

template <typename T, int TN>
void LaunchNorm(const RowProduct& p, hipStream_t stream) {
  switch ((p.k / 64 + 3) / 4) {
    case 1: LaunchRing<T, 1, TN, 4, 1>(p, stream); break;
    case 2: LaunchRing<T, 1, TN, 4, 2>(p, stream); break;
    case 3: LaunchRing<T, 1, TN, 4, 3>(p, stream); break;
    case 4: LaunchRing<T, 1, TN, 4, 4>(p, stream); break;
    default: LaunchRing<T, 1, TN, 4, 5>(p, stream); break;
  }
}

// A single row of up to 256 blocks is ahead on gemm_rows_kernel where little is left of the rings' gain: the sixteen lanes that ask for
// the one row of A there ask for the same bytes, while a ring brings them as a whole fragment; and a lane has one value for gelu there
// (0.1 us), four here (0.4 us).  us, that kernel | rings, fp16, plain: 64 -> 1024 2.3 | 2.6, 128 -> 512 2.5 | 2.6, 1024 -> 4096 3.8 | 4.1, but 1024 -> 1024
// 3.4 | 3.4, 384 -> 1536 3.0 | 2.9, 1280 -> 4096 4.9 | 4.4, 4096 -> 1024 6.9 | 4.8; gelu 128 -> 2048 2.7 | 3.1, 384 -> 1536 3.1 | 3.3, 640 -> 2560 3.5 | 3.9, 1024 -> 4096 3.9 | 4.5, but 256 ->
// 768 3.2 | 3.1, 1280 -> 3840 4.9 | 4.7; norm and gelu 1152 -> 4096 5.5 | 5.9, 1280 -> 3840 5.5 | 5.9, but 768 -> 3072 5.2 | 4.9, norm alone 1024 -> 4096 5.3 | 5.1.
// (With norm and gelu 1024 -> 4096, 5.4 | 5.5, is even: a decoding block of one row of 1024 takes 28.4 us with it there, 28.1 with it here.  Two rows: gelu 640 -> 2560 3.9 | 3.9, 256 -> 4096 3.8 | 3.6.)
bool OneRow(const RowProduct& p) {
  if (p.m != 1 || p.n > 4096) return false;
  if (p.gamma) return p.gelu && p.k > 1024;
  if (p.gelu) return p.k <= 1024 && p.k != 256;
  return p.k <= 128 || (p.k > 768 && p.k <= 1024 && p.n > 2048);
}

template <typename T>
bool TryRing(const RowProduct& p, hipStream_t stream) {
  if (!RowRingTakes(p) || OneRow(p)) return false;
  CountLaunch(kCountRowsRing);
  if (p.gamma) {
    // With a block for every CU twice the columns in each: 1 x 384 -> 6272 4.4 | 3.8, 32 x 768 -> 3072 5.5 | 4.5, 16 x 1280 -> 5120 8.8 |
    // 5.7 (its rings leave room for one block on a CU); 256 blocks 16 x 1024 -> 4096 4.7 | 5.0
    if ((p.m + 15) / 16 * ((p.n + 15) / 16) > 256) {
      LaunchNorm<T, 2>(p, stream);
    } else {
      LaunchNorm<T, 1>(p, stream);
    }
    return true;
  }
  struct Tile {
    int tm, tn, nw;
    void (*launch)(const RowProduct&, hipStream_t);
  };
  static const Tile tiles[] = {{1, 1, 8, LaunchRing<T, 1, 1, 8, 0>}, {1, 1, 4, LaunchRing<T, 1, 1, 4, 0>}, {1, 2, 4, LaunchRing<T, 1, 2, 4, 0>},
                               {2, 2, 4, LaunchRing<T, 2, 2, 4, 0>}, {2, 4, 4, LaunchRing<T, 2, 4, 4, 0>}, {4, 4, 4, LaunchRing<T, 4, 4, 4, 0>}};
  const Tile* best = nullptr;
  double best_us   = 0.0;
  for (const Tile& t : tiles) {
    const double us = few::Estimate(p.m, p.n, p.k / 64, false, t.tm, t.tn, t.nw);
    if (!best || us < best_us) best = &t, best_us = us;
  }
  best->launch(p, stream);
  return true;
}

template <typename T>
void Launch(const RowProduct& p, hipStream_t stream) {
  if (TryRing<T>(p, stream)) {
    CINN_HIP_CALL(hipGetLastError());
    return;
  }
  CountLaunch(kCountRows);
  int mt = (p.m + 15) / 16;
  dim3 grid((unsigned)((p.n + 15) / 16));
  // Fewer column blocks than CUs: one block per 16 rows as well.  A block's traffic is its 16 columns of B plus the
  // rows of A it multiplies, and with all of A (128 KB at 32 x 2048, against 64 KB of B) the few CUs at work are bound
  // by what one CU can pull in; row blocks read B again, out of L2.  ResNet-50's classifier, 32 x 2048 -> 1000: 126
  // blocks instead of 63, 2.2 us less.  With the chip full, the row tiles stay in one block's registers (B read once).
  // FLAGS_cinn_hip_gemm_skinny_rows: 0 never splits the rows, 2 always.
  static const int rows_flag = getenv("FLAGS_cinn_hip_gemm_skinny_rows") ? atoi(getenv("FLAGS_cinn_hip_gemm_skinny_rows")) : 1;
  if (p.gamma || p.gelu || rows_flag == 2 || (rows_flag == 1 && grid.x < 256)) grid.y = mt, mt = 1;
#define CINN_ROWS(MT, NORM, GELU) hipLaunchKernelGGL((gemm_rows_kernel<T, MT, NORM, GELU>), grid, dim3(64 * NW), 0, stream, p)
  // (8 x 768 x 3072 takes 6.7 us; 8.3 with sixteen wavefronts, 8.2 with all twelve k-blocks of a wavefront requested at once)
  if (p.gamma && p.gelu) {
    CINN_ROWS(1, true, true);
  } else if (p.gamma) {
    CINN_ROWS(1, true, false);
  } else if (p.gelu) {
    CINN_ROWS(1, false, true);
  } else {
    switch (mt) {
      case 1: CINN_ROWS(1, false, false); break;
      case 2: CINN_ROWS(2, false, false); break;
      case 3: CINN_ROWS(3, false, false); break;
      default: CINN_ROWS(4, false, false); break;
    }
  }
#undef CINN_ROWS
  CINN_HIP_CALL(hipGetLastError());
}

}  // namespace

bool RowProductSupported(const RowProduct& p) {
  if (p.m < 1 || p.m > 64 || p.n < 1 || p.k < 32 || p.k % 32 != 0 || (int64_t)p.n * p.k >= INT_MAX) return false;
  if (p.width < 1 || p.n % p.width != 0 || p.n / p.width > 3 || (p.n > p.width && p.residual)) return false;
  return !p.gamma || (p.beta && p.k <= kRowProductMaxNormK);
}

// whole K steps in aligned rows, results in aligned groups of four columns
bool RowRingTakes(const RowProduct& p) {
  uintptr_t wide = 0, four = 0;
  for (const void* q : {p.a, p.b, static_cast<const void*>(p.scale), static_cast<const void*>(p.shift), p.gamma, p.beta}) wide |= reinterpret_cast<uintptr_t>(q);
  for (const void* q : {p.residual, static_cast<const void*>(p.c[0]), static_cast<const void*>(p.c[1]), static_cast<const void*>(p.c[2])}) four |= reinterpret_cast<uintptr_t>(q);
  return p.k % 64 == 0 && p.n % 4 == 0 && p.width % 4 == 0 && wide % 16 == 0 && four % 8 == 0 && (int64_t)p.m * p.k < (1 << 30) && (int64_t)p.n * p.k < (1 << 30);
}

// For gemm_rows_kernel: every wavefront waits for its own rows of B: with one block per CU (16 columns each; 16 rows, or all of them from 256 blocks of
// columns on) that hides the launch, further ones take about as long again, where the tiled kernels need a few hundred tiles for
// the same result.  us, tiled | here, fp16, at most as many blocks as CUs: 16 x 192 -> 4096 3.9 | 3.8, 64 x 960 -> 1000 7.3 | 4.3, two row
// tiles in each 32 x 192 -> 4096 4.0 | 4.6, 32 x 384 -> 4096 4.7 | 4.6; two on a CU: 1 x 384 -> 8192 4.7 | 3.7, 16 x 384 -> 8192 4.8 | 5.2, 16 x 960 ->
// 8192 7.1 | 6.1, 48 x 960 -> 4096 (three row tiles) 7.3 | 6.3; three: 1 x 1984 -> 12288 12.4 | 11.5, 48 x 960 -> 3072 7.3 | 9.0, 32 x 960 -> 8192
// 7.2 | 8.0; more: 64 x 192 -> 8192 4.3 | 10.7.  Where K is no multiple of 64 the tiled kernel is the register-staged one: 1 x 1120 -> 16384 10.4 |
// 8.2, 32 x 224 -> 3072 4.9 | 4.2, 64 x 224 -> 4096 5.2 | 4.8, 32 x 544 -> 8192 6.6 | 4.9, but 32 x 2080 -> 8192 13.0 | 13.5, 48 x 224 -> 3072 5.1 | 6.1, 64 x 6112 -> 4096 and gelu 20.4 |
// 26.5.
// K in whole shares of all wavefronts has always come here.
// That kernel splits a long K over more blocks than there are columns, where it can take the product (a plain one: `splits`): 64 x 6112 -> 64
// 9.1 | 9.7, 24 x 7968 -> 200 9.1 | 11.7 (but 1 x 6112 -> 1000 8.7 | 7.0), 64 x 5024 -> 2048 11.7 | 14.9, 24 x 3968 -> 25 7.2 | 8.7; a layer with its scale
// and shift has a convolution's tiles instead, 8 x 6112 -> 4096 with gelu 18.7 | 10.0.
bool RowProductPays(int m, int n, int k, bool ring, bool saves_launch, bool splits) {
  if (ring) {
    // More than two row tiles of many columns: the tiled kernels' larger tiles pull in less, until K is long enough to be shared.  us,
    // tiled | here, fp16: 64 x 64 -> 12288 3.7 | 5.3, 64 x 512 -> 12288 5.8 | 6.4, 64 x 512 -> 32768 8.7 | 12.8, 64 x 1024 -> 32768 14.5 | 18.8, 32 x 192 ->
    // 32768 5.8 | 6.6; 64 x 128 -> 8192 3.9 | 3.9, 64 x 2048 -> 16384 15.0 | 15.2, 32 x 320 -> 32768 6.8 | 6.9, 16 x 1024 -> 8192 7.9 | 3.4.
    return saves_launch || n <= 8192 || m <= 16 || (m <= 32 && (n <= 16384 || k >= 320)) || k >= (n <= 16384 ? 1024 : 2048);
  }
  if (k % 256 == 0) return true;
  const int columns = (n + 15) / 16, tiles = (m + 15) / 16;
  const double load = columns < 256 ? (columns * tiles + 255) / 256 : (columns + 255) / 256 * (0.5 + 0.5 * tiles);
  if (splits && (k % 64 != 0 ? k >= (load > 1.0 ? 3584 : m <= 4 ? 8192 : 5632) : n % 8 != 0 && k > (m <= 4 ? 4096 : 2560))) return false;
  if (saves_launch && load <= 3.0) return true;
  if (k % 64 != 0) return load <= (m <= 4 ? 4.0 : k < 3072 ? 2.5 : 2.0) || (load <= 3.0 && (k <= 128 || k > 256) && k < 1536);
  if (m <= 4) return load <= (k < 512 ? 2.0 : 3.0);
  return load <= (k < 256 ? 1.0 : k < 512 ? 1.5 : 2.0);
}

// For gemm_rows_kernel, blocks of one row tile each: B is read for every one of them, and each normalises its rows again, so that the second and third
// round of blocks cost what a kernel of their own does - unless the product alone would be blocks of one row tile as well.  us,
// separate | inside, fp16, norm: one round 32 x 320 -> 2048 6.7 | 5.7, 64 x 960 -> 1024 10.0 | 6.1; two 32 x 384 -> 4096 7.0 | 8.5, 16 x 960 -> 8192
// 9.8 | 9.0; three 48 x 960 -> 4096 10.0 | 12.3, 48 x 1280 -> 4096 13.0 | 12.6; more 48 x 384 -> 6272 7.3 | 18.6, 64 x 1280 -> 4096 14.9 | 16.1; the
// same blocks alone 64 x 768 -> 3072 12.7 | 12.1, 48 x 512 -> 3072 10.8 | 11.8, in a
// block of a transformer (48 tokens of 512, three results) all of it 41.0 | 38.5.  gelu: two rounds 16 x 384 -> 8192 7.6 | 5.6, three 64 x 192 -> 3072
// 7.1 | 8.5, four 64 x 960 -> 4096 10.3 | 10.6, 64 x 960 -> 8192 10.8 | 20.6; the same blocks alone 64 x 768 -> 3072 12.6 | 10.3, 1 x
// 2048 -> 16384 17.1 | 14.0, but 32 x 8192 -> 4096 (alone one round of two row tiles) 26.8 | 31.5.  Both: one round
// 64 x 320 -> 1024 9.9 | 6.2, two 16 x 128 -> 8192 8.3 | 8.9, 48 x 192 -> 2048 9.2 | 8.9, three 64 x 320 -> 3072 10.0 | 12.6, six 64 x 1280 -> 6144 28.1 |
// 24.9, eight 64 x 1280 -> 8192 28.9 | 32.6, four 64 x 768 -> 4096 13.0 | 16.9; the same blocks alone 64 x 768 -> 3072 15.5 | 13.1.
RowFusion ChooseRowFusion(int m, int n, int k, bool ring, RowFusion there) {
  if (ring) {
    // gemm_rows_ring_kernel, blocks of 16 or of 32 columns; 197 layers of a program, 1 to 64 rows, us with the one outside | inside, fp16.
    // gelu is ahead everywhere, 1.09 to 1.76: 1 x 128 -> 4096 5.1 | 3.1, 64 x 768 -> 8192 9.3 | 7.4, 64 x 2048 -> 8192 12.0 | 10.3, 64 x 1280 -> 9984
    // 13.6 | 11.7.  The norm, which every block repeats for its rows, is 1.00 to 1.6 up to 512 blocks of 32 columns: 16 x 128 -> 8192 (256) 5.0 | 3.8,
    // 48 x 1280 -> 4096 (384) 9.8 | 9.3, 64 x 1024 -> 4096 (512) 8.0 | 7.8, 16 x 1280 -> 16384 (512) 13.2 | 11.3; beyond, 1.03 to 1.45 up to a K of 384 and
    // 0.76 to 1.01 from 768 on: 48 x 384 -> 6272 (588) 7.4 | 6.0, 64 x 384 -> 9984 (1248) 9.2 | 8.7; 48 x 768 -> 6272 9.4 | 9.8, 64 x 1280 -> 8192 11.9 | 15.1.
    // Even are three and four row tiles of up to 4096 columns with a K of 1024, of which the product alone has whole pairs of steps for each of its
    // wavefronts: 48 x 1024 -> 3072 7.6 | 7.6, 64 x 1024 -> 4096 8.0 | 7.8, a block of 48 tokens of 1024 31.8 | 32.2; they stay outside.
    const int tiles = (m + 15) / 16, wide = tiles * ((n + 31) / 32);
    const bool even = tiles >= 3 && n <= 4096 && k > 512 && k % 512 == 0;
    return {there.norm && (k <= 384 || (wide <= 512 && !even)), there.gelu};
  }
  const int rounds = ((n + 15) / 16 * ((m + 15) / 16) + 255) / 256;
  const bool same  = k % 256 == 0 && n <= 4080;  // the blocks of the product alone
  if (there.norm && there.gelu && (same || rounds <= 1 || (rounds <= 2 && k >= 192) || (rounds <= 6 && k >= 1152))) return there;
  if (there.gelu && ((rounds <= 2 && k < 3072) || ((n <= 4080 || m <= 16) && RowProductPays(m, n, k, false, false, false)))) return {false, true};
  return {there.norm && (rounds <= 1 || (same && k >= (rounds <= 2 ? 512 : 768)) || (rounds <= 2 && k >= 896) || (rounds <= 3 && k >= 1152)), false};
}

void RunRowProduct(const RowProduct& p, hipStream_t stream) {
  if (p.bf16) {
    Launch<__bf16>(p, stream);
  } else {
    Launch<_Float16>(p, stream);
  }
}

}  // namespace cinn_hip_kernels

extern "C" void cinn_call_hip_matmul_rows(void* v_args, int num_args, int m, int n, int k, int operands, int outputs, float epsilon,
                                          int gelu, void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  using namespace cinn_hip_kernels;
  CINN_RT_CHECK(outputs >= 1 && outputs <= 3 && num_args > outputs, "cinn_call_hip_matmul_rows: %d of %d arguments are results", outputs, num_args);
  auto* args  = static_cast<cinn_pod_value_t*>(v_args);
  auto buffer = [&](int index) {
    CINN_RT_CHECK(args[index].type_code_ == CINN_POD_BUFFER_P, "cinn_call_hip_matmul_rows: argument %d is not a buffer", index);
    auto* b = static_cast<cinn_buffer_t*>(args[index].value_.v_handle);
    CINN_RT_CHECK(b && b->memory, "cinn_call_hip_matmul_rows: argument %d has no device memory", index);
    return b;
  };
  auto operand = [&](int slot) -> cinn_buffer_t* {
    const int at = (int)(((unsigned)operands >> (4 * slot)) & 15);
    if (at == 15) return nullptr;
    CINN_RT_CHECK(at < num_args - outputs, "cinn_call_hip_matmul_rows: operand %d is argument %d of %d inputs", slot, at, num_args - outputs);
    return buffer(at);
  };
  cinn_buffer_t* in[7];
  for (int s = 0; s < 7; ++s) in[s] = operand(s);
  CINN_RT_CHECK(in[0] && in[1] && !in[5] == !in[6], "cinn_call_hip_matmul_rows: x and W, and gamma and beta or neither, expected");
  const cinn_type_t type = in[0]->type;
  RowProduct p{};
  p.bf16 = type.code == cinn_type_bfloat;
  CINN_RT_CHECK(type.bits == 16 && (p.bf16 || type.code == cinn_type_float), "cinn_call_hip_matmul_rows: fp16 or bf16 operands expected");
  for (int s : {1, 4, 5, 6})
    CINN_RT_CHECK(!in[s] || (in[s]->type.code == type.code && in[s]->type.bits == 16), "cinn_call_hip_matmul_rows: operand %d differs in type", s);
  for (int s : {2, 3})
    CINN_RT_CHECK(!in[s] || (in[s]->type.code == cinn_type_float && in[s]->type.bits == 32), "cinn_call_hip_matmul_rows: scale and shift are fp32");
  auto memory = [&](int slot) -> void* { return in[slot] ? in[slot]->memory : nullptr; };
  p.a = memory(0), p.b = memory(1);
  p.scale = static_cast<const float*>(memory(2)), p.shift = static_cast<const float*>(memory(3));
  p.alpha    = 1.0f;
  p.residual = memory(4), p.residual_scale = 1.0f;
  p.gamma = memory(5), p.beta = memory(6), p.epsilon = epsilon;
  p.gelu = gelu != 0;
  p.m = m, p.n = n, p.k = k;
  CINN_RT_CHECK(n > 0 && n % outputs == 0, "cinn_call_hip_matmul_rows: %d columns for %d results", n, outputs);
  p.width = n / outputs;
  for (int i = 0; i < outputs; ++i) {
    cinn_buffer_t* out = buffer(num_args - outputs + i);
    CINN_RT_CHECK(out->type.code == type.code && out->type.bits == 16, "cinn_call_hip_matmul_rows: result %d differs in type", i);
    p.c[i] = out->memory;
  }
  CINN_RT_CHECK(RowProductSupported(p), "cinn_call_hip_matmul_rows: %d x %d x %d is not taken", m, n, k);
  RunRowProduct(p, static_cast<hipStream_t>(stream));
}
