// Register-staged MFMA matrix product for gfx950: any extents, any operand layout, any alignment, fp16 / bf16 / fp32.
//
//   C[m][n] = epilogue( sum_k A[m][k] B[k][n] ),  A stored [m][k] or [k][m], B stored [n][k] or [k][n]
//
// The direct-to-LDS kernels of gemm_mfma.hip need whole, aligned 16-byte chunks and enough tiles.  Everything else comes
// here: extents that are no multiple of anything, few tiles, many small batch entries.  What it does instead:
//   * an operand keeps its own order on the way into LDS: a K-contiguous one as [row][128 bytes of k], the other as
//     [k][rows].  Fragments of the latter are read with ds_read_b64_tr_b16 (16-bit) or as single floats, so nothing is
//     transposed in registers or in memory beforehand;
//   * chunks travel global -> registers -> LDS, one K step ahead: a global load takes any element-aligned address and a
//     chunk can be masked.  Chunks that reach beyond K, or beyond the end of the operand's last row, only occur in the
//     last step or two of a product; those run a guarded loader, all others an unguarded one;
//   * rows beyond M / N repeat the last one; what they produce is not stored;
//   * grids too small for the chip split K over blockIdx.z, and a second kernel adds the fp32 planes.
// Measured before (transposing copies in front of a convolution kernel, one launch per batch entry, or scalar FMAs
// where K was no multiple of a chunk) and here, us: fp16 A^T B 768 x 3072 x 4100 871 -> 39 (direct-to-LDS 28.5), [64] x 1 x 215
// x 48 262 -> 4.0, 1000^3 15.3 -> 10.4; bf16 [2] x 2336 x 3250 x 153 120 -> 25, 512 x 512 x 4096 26 -> 14; fp32 1000^3
// 36 -> 24 (84 TFLOP/s), A^T B 768 x 3072 x 4100 218 -> 171 (113 TFLOP/s).  A step of a 64x64 tile is bound by the trip of its chunks to LDS
// (0.42 us for a block alone), of a 128x128 tile by the register staging around its MFMAs (0.6 us for 0.2 of MFMA).
#include "kernels/gemm_flex.h"

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <type_traits>

#include "kernels/flex_tile.h"
#include "kernels/launch_count.h"
#include "runtime/hip_check.h"
#include "runtime/scratch.h"

namespace cinn_hip_kernels {
namespace {

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
  const float* shift;
  const void* residual;
  float alpha, residual_scale;
  const void* shift16;  // the shift in the matrices' 16-bit type (last: in front of the others it cost the fp32 products 2%)
};

// `residual` is 0 where there is none
__device__ __forceinline__ float Finish(float v, float alpha, float shift, float residual_scale, float residual) {
  return __builtin_fmaf(residual_scale, residual, __builtin_fmaf(v, alpha, shift));
}

// KG groups of four wavefronts (2 x 2 over the tile) share the block's tiles and take a K step's slices in turn; their
// sums meet in the epilogue.
// Block `bid` of the tiles, `z` of the splits, batch entry `entry` of `entries`.
template <typename T, bool A_KC, bool B_KC, int BM, int BN, int KG, int PARTS = 0>
__device__ __forceinline__ void FlexBlock(const FlexParams& p, char* lds, int bid, int z, int entry, int entries) {
  const int tid = threadIdx.x;
  int tm, tn;
  flex::TileOf(bid, p.tiles_m, p.tiles_n, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN;

  flex::Tile<T, A_KC, BM, 256 * KG> ta;
  flex::Tile<T, B_KC, BN, 256 * KG> tb;
  ta.Init(static_cast<const T*>(p.a) + entry * p.stride_a, p.lda, m0, p.m, p.k, tid);
  tb.Init(static_cast<const T*>(p.b) + entry * p.stride_b, p.ldb, n0, p.n, p.k, tid);
  typename flex::Mma<T, A_KC, B_KC, BM, BN>::acc_t acc;
  const int s0 = z * p.steps_per_split;
  flex::KLoop<T, A_KC, B_KC, BM, BN, KG, PARTS>(lds, ta, tb, s0, min(s0 + p.steps_per_split, p.steps), p.full_steps, p.k, tid, acc);

  const int col0 = n0 + tid % (BN / 8) * 8;  // the eight columns this thread finishes
  const int cols = min(p.n - col0, 8);
  float sh[8];
  if (!p.partials) {
#pragma unroll
    for (int e = 0; e < 8; ++e) sh[e] = p.shift ? p.shift[min(col0 + e, p.n - 1)] : 0.0f;
    if (sizeof(T) == 2 && p.shift16) {
#pragma unroll
      for (int e = 0; e < 8; ++e) sh[e] = (float)static_cast<const T*>(p.shift16)[min(col0 + e, p.n - 1)];
    }
  }
  T* c              = static_cast<T*>(p.c) + entry * p.stride_c;
  const T* residual = p.residual ? static_cast<const T*>(p.residual) + entry * p.stride_c : nullptr;
  float* plane      = p.partials + ((int64_t)z * entries + entry) * p.m * p.n;
  flex::EachRowGroup<T, A_KC, B_KC, BM, BN, KG>(lds, acc, tid, [&](int row, int, const float (&v)[8]) {
    const int m = m0 + row;
    if (m >= p.m || cols <= 0) return;
    const int64_t at = (int64_t)m * p.n + col0;
    if (p.partials) {
      if (cols == 8) {
        __builtin_memcpy(plane + at, v, 32);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (e < cols) plane[at + e] = v[e];
      }
      return;
    }
    if (cols == 8) {
      typedef T vec8 __attribute__((ext_vector_type(8)));
      vec8 out, res = {0, 0, 0, 0, 0, 0, 0, 0};
      if (residual) __builtin_memcpy(&res, residual + at, 8 * sizeof(T));
#pragma unroll
      for (int e = 0; e < 8; ++e) out[e] = (T)Finish(v[e], p.alpha, sh[e], p.residual_scale, (float)res[e]);
      __builtin_memcpy(c + at, &out, 8 * sizeof(T));
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < cols)
          c[at + e] = (T)Finish(v[e], p.alpha, sh[e], p.residual_scale, residual ? (float)residual[at + e] : 0.0f);
    }
  });
}

template <typename T, bool A_KC, bool B_KC, int BM, int BN, int KG>
__global__ void __launch_bounds__(256 * KG, 2)
flex_gemm_kernel(FlexParams p) {
  __shared__ __attribute__((aligned(256))) char lds[2 * (BM + BN) * 128];
  FlexBlock<T, A_KC, B_KC, BM, BN, KG>(p, lds, blockIdx.x, blockIdx.z, blockIdx.y, gridDim.y);
}

// Several products on 64x64 tiles.  A layer's y, dx and dW are three products of the same volume, which each took a launch and
// mostly one more to add the partial sums of a split K, because none has the tiles for all CUs by itself: small ones are bound by
// those launches (about 3 us each), larger ones by their nearly empty rounds.  Together they share the CUs and one addition.  us of
// the step with its two column sums, one by one | together: 37 x 75 -> 247 fp16 19.8 | 9.4, 665 x 233 -> 670 bf16 28.5 | 13.9,
// 874 x 1237 -> 440 fp32 68 | 53, 630 x 2558 -> 1999 bf16 88 | 67.
// Blocks [first[i], first[i + 1]) are product i's, split by split, the tiles of each in whole rounds of the XCDs (what is beyond
// them returns at once): TileOf's neighbours stay on one XCD.
struct GroupParams {
  FlexParams p[kFlexGroup];
  int first[kFlexGroup + 1];
  int layout[kFlexGroup];  // bit 0: a_kc, bit 1: b_kc
  int count;
};

__device__ __forceinline__ int MemberOf(const int* first, int count, int bid) {
  int i = 0;
  while (i + 1 < count && bid >= first[i + 1]) ++i;
  return i;
}

template <typename T>
__global__ void __launch_bounds__(256, 2)
flex_group_kernel(GroupParams g) {
  __shared__ __attribute__((aligned(256))) char lds[2 * 128 * 128];
  const int i         = MemberOf(g.first, g.count, blockIdx.x);
  const FlexParams& p = g.p[i];
  const int tiles = p.tiles_m * p.tiles_n, round = (tiles + 7) & ~7, at = (int)blockIdx.x - g.first[i];
  const int z = at / round, bid = at - z * round;
  if (bid >= tiles) return;
  // fp32: the sums of a K step before they are added to those of the others, as a block may have more steps here than alone.
  // Relative error against float64, 27 products of small layers: up to 1.5 times of the separate ones' as one chain, 0.51 on average so and
  // nowhere more.  50.2 -> 53.2 us at 874 x 1237 -> 440.
  constexpr int kParts = sizeof(T) == 4 ? 1 : 0;
  switch (g.layout[i]) {
    case 0: FlexBlock<T, false, false, 64, 64, 1, kParts>(p, lds, bid, z, 0, 1); break;
    case 1: FlexBlock<T, true, false, 64, 64, 1, kParts>(p, lds, bid, z, 0, 1); break;
    case 2: FlexBlock<T, false, true, 64, 64, 1, kParts>(p, lds, bid, z, 0, 1); break;
    default: FlexBlock<T, true, true, 64, 64, 1, kParts>(p, lds, bid, z, 0, 1); break;
  }
}

// Adds the planes of a split reduction and applies the epilogue: one thread per V consecutive elements of a plane row
// (V divides n), planes in ascending order.
template <typename T, int V>
__device__ __forceinline__ void ReduceBlock(const FlexParams& p, int splits, int64_t plane, int bid) {
  const int64_t at = ((int64_t)bid * 256 + threadIdx.x) * V;
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
  float sh[V];
#pragma unroll
  for (int e = 0; e < V; ++e) res[e] = (T)0.0f, sh[e] = p.shift ? p.shift[col + e] : 0.0f;
  if (sizeof(T) == 2 && p.shift16) {
#pragma unroll
    for (int e = 0; e < V; ++e) sh[e] = (float)static_cast<const T*>(p.shift16)[col + e];
  }
  if (p.residual) __builtin_memcpy(res, static_cast<const T*>(p.residual) + at, V * sizeof(T));
#pragma unroll
  for (int e = 0; e < V; ++e)
    out[e] = (T)Finish(v[e], p.alpha, sh[e], p.residual_scale, (float)res[e]);
  __builtin_memcpy(static_cast<T*>(p.c) + at, out, V * sizeof(T));
}

template <typename T, int V>
__global__ void __launch_bounds__(256)
flex_reduce_kernel(FlexParams p, int splits, int64_t plane) {
  ReduceBlock<T, V>(p, splits, plane, blockIdx.x);
}

template <typename T>
__global__ void __launch_bounds__(256)
flex_group_reduce_kernel(GroupParams g) {
  const int i         = MemberOf(g.first, g.count, blockIdx.x);
  const FlexParams& p = g.p[i];
  const int splits = (p.steps + p.steps_per_split - 1) / p.steps_per_split, bid = (int)blockIdx.x - g.first[i];
  if (p.n % 4 == 0) {
    ReduceBlock<T, 4>(p, splits, (int64_t)p.m * p.n, bid);
  } else {
    ReduceBlock<T, 1>(p, splits, (int64_t)p.m * p.n, bid);
  }
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

// the partial sums of a split
size_t PlaneBytes(const FlexGemm& g, int splits) { return (size_t)splits * g.batch * g.m * g.n * sizeof(float); }

// Block tile and K split with the smallest estimated time.  The estimate (us) adds, per CU, the K steps of the blocks
// it gets, and what a split writes and reads back.  A block alone on its CU takes `alone` per step, blocks that share
// one take `shared` each, at most `resident` at a time; its start and epilogue are worth `extra` steps, which decides
// short reductions.  Fitted to every tile at M = N = 1600, 2056, 3000, 4000 and 1000 x 3000 with K = 40 to 4000 (16 bits).
// us on 64x64 | 128x128 | 128x128 tiles of two groups: 3000 x 3000 x 200 17.7 | 17.8 | 27.2 (with two steps' worth for every
// tile, as the estimate once had it, the last was chosen), x 4000 134 | 137 | 119; 1600 x 1600 x 200 7.8 | 8.9 | 10.1, x 1000
// 17.0 | 18.1 | 15.9; 4000 x 4000 x 4000 234 | 152 | 165; A^T B 768 x 3072 x 4100 46 | - | 39.  fp32 768 x 3072 x 4100 262 us on
// 128x128 tiles, 205 on 64x64 and 170 with K split four ways: a step is bound by the matrix pipe there, and small tiles
// spread evenly.
FlexPlan ChoosePlan(const FlexGemm& g, int steps, hipStream_t stream) {
  struct Shape {
    int tile, kg, resident;
    double alone, shared, extra;
  };
  static const Shape k16[] = {{64, 1, 4, 0.42, 0.245, 3.0}, {128, 1, 2, 0.87, 0.55, 4.0}, {128, 2, 1, 0.53, 0.53, 10.0}};
  static const Shape k32[] = {{64, 1, 4, 0.62, 0.50, 2.0}};
  const bool fp32    = g.type == FlexType::kF32;
  const Shape* shape = fp32 ? k32 : k16;
  const int shapes   = fp32 ? 1 : 3;
  const double plane = (double)g.batch * g.m * g.n;
  FlexPlan best{64, 1, 1, 1e30};
  for (int i = 0; i < shapes; ++i) {
    const Shape& t = shape[i];
    const double tiles = (double)((g.m + t.tile - 1) / t.tile) * ((g.n + t.tile - 1) / t.tile) * g.batch;
    for (int splits = 1; splits <= 16 && (splits == 1 || steps / splits >= 4); ++splits) {
      const int per_cu    = (int)((tiles * splits + 255) / 256);
      const int rounds    = per_cu / t.resident, rest = per_cu % t.resident;
      const double round  = std::max(t.alone, t.shared * t.resident);
      const double a_step = rounds * round + (rest ? std::max(t.alone, t.shared * rest) : 0.0);
      double us = a_step * ((steps + splits - 1) / splits + t.extra);
      if (splits > 1) us += 4.0 + splits * plane * 8.0 / 4e6;
      if (us < best.us) best = {t.tile, t.kg, splits, us};
    }
  }
  // under capture without an eager run or a reservation: K whole, which needs no scratch
  if (best.splits > 1 && PlaneBytes(g, best.splits) > ScratchLimit(ScratchKind::kSplitK, stream)) best.splits = 1;
  return best;
}

int Steps(const FlexGemm& g) {
  const int ks = g.type == FlexType::kF32 ? 32 : 64;
  return (g.k + ks - 1) / ks;
}

// a thread's chunk is a 32-bit byte offset from the tile's first element: 128 rows, or 64 k rows, of the operand
bool Fits(const FlexGemm& g) {
  const int64_t limit = ((int64_t)1 << 31) / (128 * (g.type == FlexType::kF32 ? 4 : 2));
  const int64_t tiles = (int64_t)((g.m + 63) / 64) * ((g.n + 63) / 64);
  return g.lda < limit && g.ldb < limit && tiles < INT_MAX / 8 && g.batch <= 65535;
}

template <typename T, bool A_KC, bool B_KC>
void LaunchTiles(const FlexPlan& plan, dim3 grid, const FlexParams& p, hipStream_t stream) {
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

// everything but the partial sums' place; `plan.splits` becomes the splits that there are
template <typename T>
FlexParams ParamsOf(const FlexGemm& g, FlexPlan* plan) {
  FlexParams p;
  p.a = g.a, p.b = g.b, p.c = g.c;
  p.m = g.m, p.n = g.n, p.k = g.k;
  p.lda = g.lda, p.ldb = g.ldb;
  p.stride_a = g.stride_a, p.stride_b = g.stride_b, p.stride_c = g.stride_c;
  p.steps      = Steps(g);
  p.full_steps = std::min(FullSteps<T>(g.a_kc, g.lda, g.m, g.k), FullSteps<T>(g.b_kc, g.ldb, g.n, g.k));
  p.shift = g.shift, p.shift16 = g.shift16, p.residual = g.residual;
  p.alpha = g.alpha, p.residual_scale = g.residual_scale;
  p.steps_per_split = (p.steps + plan->splits - 1) / plan->splits;
  plan->splits      = (p.steps + p.steps_per_split - 1) / p.steps_per_split;
  p.tiles_m         = (g.m + plan->tile - 1) / plan->tile;
  p.tiles_n         = (g.n + plan->tile - 1) / plan->tile;
  p.partials        = nullptr;
  return p;
}

template <typename T>
void Launch(const FlexGemm& g, FlexPlan plan, hipStream_t stream) {
  FlexParams p        = ParamsOf<T>(g, &plan);
  const int64_t plane = (int64_t)g.batch * g.m * g.n;
  if (plan.splits > 1) p.partials = static_cast<float*>(Scratch(ScratchKind::kSplitK, PlaneBytes(g, plan.splits), stream));
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

template <typename T>
void LaunchGroup(const FlexGemm* g, const int* splits, int count, hipStream_t stream) {
  GroupParams group;
  group.count = count;
  size_t bytes = 0, at[kFlexGroup];
  int blocks = 0;
  for (int i = 0; i < count; ++i) {
    FlexPlan plan{64, 1, splits[i], 0.0};
    group.p[i]      = ParamsOf<T>(g[i], &plan);
    group.layout[i] = (g[i].a_kc ? 1 : 0) | (g[i].b_kc ? 2 : 0);
    group.first[i]  = blocks;
    blocks += (group.p[i].tiles_m * group.p[i].tiles_n + 7) / 8 * 8 * plan.splits;
    at[i] = SIZE_MAX;
    if (plan.splits > 1) at[i] = bytes, bytes += (PlaneBytes(g[i], plan.splits) + 255) / 256 * 256;
  }
  group.first[count] = blocks;
  if (bytes) {
    char* planes = static_cast<char*>(Scratch(ScratchKind::kSplitK, bytes, stream));
    for (int i = 0; i < count; ++i)
      if (at[i] != SIZE_MAX) group.p[i].partials = reinterpret_cast<float*>(planes + at[i]);
  }
  hipLaunchKernelGGL((flex_group_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, stream, group);
  if (bytes) {
    GroupParams reduce;
    reduce.count = 0;
    blocks       = 0;
    for (int i = 0; i < count; ++i) {
      if (!group.p[i].partials) continue;
      reduce.p[reduce.count]       = group.p[i];
      reduce.first[reduce.count++] = blocks;
      const int64_t threads = (int64_t)g[i].m * g[i].n / (g[i].n % 4 == 0 ? 4 : 1);
      blocks += (int)((threads + 255) / 256);
    }
    reduce.first[reduce.count] = blocks;
    hipLaunchKernelGGL((flex_group_reduce_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, stream, reduce);
  }
  CINN_HIP_CALL(hipGetLastError());
}

}  // namespace

bool PlanFlexGemm(const FlexGemm& g, hipStream_t stream, FlexPlan* plan) {
  if (!Fits(g)) return false;
  *plan = ChoosePlan(g, Steps(g), stream);
  return true;
}

void RunFlexGemm(const FlexGemm& g, FlexPlan plan, hipStream_t stream) {
  switch (g.type) {
    case FlexType::kF16: Launch<_Float16>(g, plan, stream); break;
    case FlexType::kBF16: Launch<__bf16>(g, plan, stream); break;
    case FlexType::kF32: Launch<float>(g, plan, stream); break;
  }
}

// The split of a group: all products with at most the same number of K steps in a block, the number that the model of ChoosePlan
// likes best.  Against the sum of the separate estimates one tenth is asked for.  Over 70 linear layers' steps (y, dx and dW; 32 to
// 12950 rows of 65 to 3989 values, the three types) all whose estimate was that far below were faster together, by 1.14 to 2.1.
// Those above it were about even (68 | 65 us at 12950 x 108 -> 1200 in fp16, 91 | 81 at 7863 x 1533 -> 116) or slower (96 | 119 at
// 4887 x 301 -> 2123): large products have 128x128 tiles by themselves.
bool TryFlexGroup(const FlexGemm* g, const FlexPlan* alone, int count, hipStream_t stream) {
  static const bool enabled = !(getenv("FLAGS_cinn_hip_gemm_group") && atoi(getenv("FLAGS_cinn_hip_gemm_group")) == 0);
  if (!enabled || count < 2 || count > kFlexGroup) return false;
  const bool fp32 = g[0].type == FlexType::kF32;
  int longest = 0;
  double sum = 0.0;
  for (int i = 0; i < count; ++i) {
    if (g[i].type != g[0].type || g[i].batch != 1 || !Fits(g[i])) return false;
    longest = std::max(longest, Steps(g[i]));
    sum += alone[i].us;
  }
  const double one = fp32 ? 0.62 : 0.42, shared = fp32 ? 0.50 : 0.245, start = fp32 ? 2.0 : 3.0;  // as in ChoosePlan
  const size_t room = ScratchLimit(ScratchKind::kSplitK, stream);
  int splits[kFlexGroup] = {1, 1, 1, 1};
  double best = 1e30;
  for (int most = longest;;) {
    int s[kFlexGroup], block = 0;
    double steps = 0.0, bytes = 0.0, blocks = 0.0;
    size_t planes = 0;
    for (int i = 0; i < count; ++i) {
      const int all = Steps(g[i]);
      const double tiles = (double)((g[i].m + 63) / 64) * ((g[i].n + 63) / 64);
      s[i]            = std::min(16, (all + most - 1) / most);
      const int share = (all + s[i] - 1) / s[i];
      block = std::max(block, share);
      blocks += (tiles + 7) * s[i];
      steps += tiles * s[i] * (share + start);
      if (s[i] > 1) bytes += 8.0 * s[i] * g[i].m * g[i].n, planes += (PlaneBytes(g[i], s[i]) + 255) / 256 * 256;
    }
    // the CUs' throughput and half of the last round, or the longest block by itself
    double us = std::max(steps / 256 * shared + 0.5 * block * shared, (block + start) * one);
    if (bytes > 0.0) us += 4.0 + bytes / 4e6;
    if (planes <= room && blocks < 1e9 && us < best) {
      best = us;
      std::copy(s, s + count, splits);
    }
    if (most <= 4) break;
    most = std::max(4, most > 8 ? most * 3 / 4 : most - 1);
  }
  if (best >= 0.9 * sum) return false;
  CountLaunch(kCountProductGroup);
  // the longest blocks first
  FlexGemm ordered[kFlexGroup];
  int order[kFlexGroup] = {0, 1, 2, 3}, ordered_splits[kFlexGroup];
  auto share = [&](int i) { return (Steps(g[i]) + splits[i] - 1) / splits[i]; };
  std::stable_sort(order, order + count, [&](int x, int y) { return share(x) > share(y); });
  for (int i = 0; i < count; ++i) ordered[i] = g[order[i]], ordered_splits[i] = splits[order[i]];
  switch (g[0].type) {
    case FlexType::kF16: LaunchGroup<_Float16>(ordered, ordered_splits, count, stream); break;
    case FlexType::kBF16: LaunchGroup<__bf16>(ordered, ordered_splits, count, stream); break;
    case FlexType::kF32: LaunchGroup<float>(ordered, ordered_splits, count, stream); break;
  }
  return true;
}

}  // namespace cinn_hip_kernels
