// Channels-last convolutions of few output tiles for gfx950: one image, or a few, through a network's deeper stages.
//
//   y[pixel][oc] = act( sum_k im2col(x)[pixel][k] w[oc][k] * scale + shift + residual ),  fp16 / bf16 / fp32
//
// The tiled kernels give such a layer 26 to 104 blocks of 64x64, split K over more blocks and add the parts in a second
// launch.  What bounds it is none of the chip's rates but one block's chain: launch, first operands, K steps with a block
// barrier each, partial sums to memory, launch, partial sums back.  Here the wavefronts of a block split K among themselves and
// the parts meet in LDS, so that a layer is one launch of small output tiles, a block for most CUs.  No operand is shared
// between wavefronts: each has a ring of K steps of its own in LDS, filled by direct global -> LDS loads, waits for nobody and
// meets the others once, at the end.
//
// What bounds it then is what one CU pulls in.  That depends on the order of a load's lanes: sixteen-byte pieces of one 128-byte
// line in eight neighbouring lanes arrive at 125 GB/s per CU (operands in L2), the same bytes in the order of an MFMA
// fragment (sixteen rows in neighbouring lanes) at 37 GB/s, which is why fragments do not come straight from memory here: the
// same kernel with its fragments loaded into registers took 6.55 us for 256 -> 256 3x3 on 14x14.  us, tiled kernels | here, fp16, one
// image, weights in the last-level cache: 128 -> 128 3x3 on 28x28 9.2 | 3.8, 256 -> 256 3x3 on 14x14 9.6 | 4.1, 1024 -> 256 1x1 7.6 | 3.4,
// 512 -> 512 3x3 on 7x7 10.5 | 5.2; fp32 15.1 | 6.5, 12.3 | 4.6, 20.9 | 9.7.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <type_traits>

#include "kernels/conv_nhwc.h"
#include "runtime/hip_check.h"
#include "runtime/scratch.h"

namespace cinn_hip_kernels {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kStepBytes = 128;  // of a row, per K step

struct FewParams {
  const void* x;
  const void* w;
  void* y;
  const float* scale;
  const float* shift;
  const void* residual;
  const void* zeros;      // 128 bytes, where a window reaches beyond the image
  int h, w_in, c;
  int oc, pixels;
  int kw;
  int pad_h, pad_w, stride_h, stride_w, dil_h, dil_w;
  int steps, steps_per_tap;  // K steps
  int tiles_m, tiles_n;
  int pixels_outer;       // neighbouring blocks of an XCD share a tile row's pixels (or a tile column's filter rows)
  unsigned magic_plane, shift_plane, magic_ow, shift_ow;
  int oh_ow, ow;
  int relu;
  float alpha, residual_scale;
};

__device__ __forceinline__ int Quotient(int n, unsigned magic, unsigned shift) {
  return (int)(((unsigned long long)(unsigned)n * magic) >> shift);
}

// 16 bytes of a filter row and of a pixel, in each of four lane groups: one 16x16x32 product, or four of 16x16x4.  The result
// has channels as its rows: a lane ends up with four consecutive channels (4 (lane / 16) ..) of pixel lane % 16.
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

// TM x TN fragments of 16 pixels x 16 channels, NW wavefronts that share K, DEPTH K steps of each in flight.
template <typename T, int TM, int TN, int NW, int DEPTH>
__global__ void __launch_bounds__(64 * NW)
conv_few_kernel(FewParams p) {
  constexpr int E     = (int)sizeof(T);
  constexpr int FRAG  = 16 * kStepBytes;           // 16 rows of a K step
  constexpr int SLOT  = (TM + TN) * FRAG;
  constexpr int RING  = DEPTH * SLOT;              // of a wavefront
  constexpr int LOADS = 2 * (TM + TN);             // of a step, 8 rows each
  static_assert(NW * RING <= 160 * 1024 && TM * TN * 1024 <= RING && DEPTH == 2 && DEPTH * LOADS < 64, "");
  __shared__ __attribute__((aligned(1024))) char lds[NW * RING];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* const ring = lds + wave * RING;
  const unsigned ring_at = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) char*)ring);
  // consecutive block ids go round-robin to the 8 XCDs: every XCD gets a contiguous run of tiles
  const int tiles = p.tiles_m * p.tiles_n, q = tiles >> 3, rest = tiles & 7, xcd = blockIdx.x & 7;
  const int id = xcd * q + min(xcd, rest) + (blockIdx.x >> 3);
  const int tm = p.pixels_outer ? id / p.tiles_n : id % p.tiles_m;
  const int tn = p.pixels_outer ? id % p.tiles_n : id / p.tiles_m;
  const int m0 = tm * (16 * TM), n0 = tn * (16 * TN);

  // A load brings 8 rows of 128 bytes, eight lanes to a row; chunk c of row r goes to place PlaceOf(c, r), which the lane's
  // choice of its chunk decides.
  int y0[2 * TM], x0[2 * TM];  // top left corner of the lane's pixels' windows
  unsigned off[2 * TM];        // byte offset of the lane's chunk there, modulo 2^32
  unsigned w_off[2 * TN];
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i) {
    const int row   = 8 * (i & 1) + (lane >> 3);
    const int chunk = ChunkAt(lane & 7, row) << 4;
    const int pixel = min(m0 + 8 * i + (lane >> 3), p.pixels - 1);  // beyond the last pixel: that one, not stored
    const int n = Quotient(pixel, p.magic_plane, p.shift_plane), in = pixel - n * p.oh_ow;
    const int oy = Quotient(in, p.magic_ow, p.shift_ow), ox = in - oy * p.ow;
    y0[i]  = oy * p.stride_h - p.pad_h;
    x0[i]  = ox * p.stride_w - p.pad_w;
    off[i] = (unsigned)((n * p.h + y0[i]) * p.w_in + x0[i]) * (unsigned)(p.c * E) + chunk;
  }
#pragma unroll
  for (int j = 0; j < 2 * TN; ++j) {
    const int row   = 8 * (j & 1) + (lane >> 3);
    const int chunk = ChunkAt(lane & 7, row) << 4;
    w_off[j]        = (unsigned)min(n0 + 8 * j + (lane >> 3), p.oc - 1) * (unsigned)(p.steps * kStepBytes) + chunk;
  }
  // what the epilogue reads: wavefront w finishes fragments w, w + NW, ...; a lane has four channels of one pixel
  constexpr int FINISH = (TM * TN + NW - 1) / NW;
  typedef T vec4 __attribute__((ext_vector_type(4)));
  f32x4 sc[FINISH], sh[FINISH];
  vec4 res[FINISH];
#pragma unroll
  for (int f = 0; f < FINISH; ++f) {
    const int frag = wave + f * NW, i = frag / TN, j = frag - i * TN;
    const int pixel = m0 + 16 * i + (lane & 15), col = n0 + 16 * j + (lane >> 4) * 4;
    const bool mine = frag < TM * TN && pixel < p.pixels && col < p.oc;
    sc[f]  = f32x4{p.alpha, p.alpha, p.alpha, p.alpha};
    sh[f]  = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    res[f] = vec4{(T)0.0f, (T)0.0f, (T)0.0f, (T)0.0f};
    if (mine && p.scale) sc[f] = *reinterpret_cast<const f32x4*>(p.scale + col);
    if (mine && p.shift) sh[f] = *reinterpret_cast<const f32x4*>(p.shift + col);
    if (mine && p.residual) res[f] = *reinterpret_cast<const vec4*>(static_cast<const T*>(p.residual) + (int64_t)pixel * p.oc + col);
  }

  // this wavefront's K steps, and the tap and channels of the next one to be requested
  const int s0 = p.steps * wave / NW, s1 = p.steps * (wave + 1) / NW;
  const int tap = s0 / p.steps_per_tap;
  int next = s0, in_tap = s0 - tap * p.steps_per_tap, dy = tap / p.kw, dx = tap - dy * p.kw;
  auto request = [&](int slot) {
    const unsigned to = ring_at + slot * SLOT;
#pragma unroll
    for (int j = 0; j < 2 * TN; ++j)
      CopyAt(to + (2 * TM + j) * (FRAG / 2), static_cast<const char*>(p.w) + (int64_t)next * kStepBytes, w_off[j]);
    const unsigned tap_at = (unsigned)((dy * p.dil_h) * p.w_in + dx * p.dil_w) * (unsigned)(p.c * E) + (unsigned)(in_tap * kStepBytes);
#pragma unroll
    for (int i = 0; i < 2 * TM; ++i) {
      const bool inside = (unsigned)(y0[i] + dy * p.dil_h) < (unsigned)p.h && (unsigned)(x0[i] + dx * p.dil_w) < (unsigned)p.w_in;
      CopyAt(to + i * (FRAG / 2), inside ? static_cast<const char*>(p.x) + (off[i] + tap_at) : static_cast<const char*>(p.zeros) + ((lane & 7) << 4));
    }
    if (++in_tap == p.steps_per_tap) {
      in_tap = 0;
      if (++dx == p.kw) dx = 0, ++dy;
    }
    ++next;
  };
  const int fr = lane & 15;
  int at[2];
#pragma unroll
  for (int half = 0; half < 2; ++half) at[half] = fr * kStepBytes + (PlaceOf(half * 4 + (lane >> 4), fr) << 4);
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  u32x4 xs[TM][2], ws[TN][2];
  auto read = [&](int slot) {
    const char* from = ring + slot * SLOT;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int j = 0; j < TN; ++j) ws[j][half] = *reinterpret_cast<const u32x4*>(from + (TM + j) * FRAG + at[half]);
#pragma unroll
      for (int i = 0; i < TM; ++i) xs[i][half] = *reinterpret_cast<const u32x4*>(from + i * FRAG + at[half]);
    }
  };
  auto multiply = [&]() {
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = Multiply<T>(ws[j][half], xs[i][half], acc[i][j]);
  };
  if (s1 - s0 >= DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) request(d);
    int s = s0;
    for (; s + 2 * DEPTH <= s1; s += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        WaitLoads<(DEPTH - 1) * LOADS>();
        read(d);
        WaitLdsReads();  // the slot is free
        request(d);
        multiply();
      }
    }
    // fewer than 2 DEPTH steps are left, DEPTH of them requested
    const int more = s1 - s - DEPTH;
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d) {
      if (d >= more) break;
      WaitLoads<(DEPTH - 1) * LOADS>();
      read(d);
      WaitLdsReads();
      request(d);
      multiply();
    }
    s += more;
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (d == 0) WaitLoads<(DEPTH - 1) * LOADS>();
      if (d == DEPTH - 1) WaitLoads<0>();
      read((more + d) % DEPTH);
      multiply();
    }
  } else {
    for (int d = 0; d < s1 - s0; ++d) request(d);
    WaitLoads<0>();
    for (int d = 0; d < s1 - s0; ++d) {
      read(d);
      multiply();
    }
  }
  // the parts meet in LDS: every wavefront's where its ring was
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) *reinterpret_cast<f32x4*>(ring + (i * TN + j) * 1024 + lane * 16) = acc[i][j];
  __syncthreads();
#pragma unroll
  for (int f = 0; f < FINISH; ++f) {
    const int frag = wave + f * NW, i = frag / TN, j = frag - i * TN;
    const int pixel = m0 + 16 * i + fr, col = n0 + 16 * j + (lane >> 4) * 4;
    if (frag >= TM * TN || pixel >= p.pixels || col >= p.oc) continue;
    f32x4 sum = *reinterpret_cast<const f32x4*>(lds + frag * 1024 + lane * 16);
#pragma unroll
    for (int k = 1; k < NW; ++k) sum += *reinterpret_cast<const f32x4*>(lds + k * RING + frag * 1024 + lane * 16);
    vec4 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = __builtin_fmaf(sum[e], sc[f][e], sh[f][e]);
      if (p.residual) v = __builtin_fmaf(p.residual_scale, (float)res[f][e], v);
      asm volatile("" : "+v"(v));  // fp32 first, then one rounding to T
      out[e] = (T)(p.relu ? fmaxf(v, 0.0f) : v);
    }
    *reinterpret_cast<vec4*>(static_cast<T*>(p.y) + (int64_t)pixel * p.oc + col) = out;
  }
}

// q = (n * magic) >> shift == n / d for 0 <= n < 2^31
void MagicFor(int d, unsigned* magic, unsigned* shift) {
  int l = 0;
  while ((1ll << l) < d) ++l;
  *shift = d == 1 ? 0 : 31 + l;
  *magic = d == 1 ? 1 : (unsigned)(((1ull << *shift) / (unsigned)d) + 1);
}

template <typename T, int TM, int TN, int NW, int DEPTH>
void Launch(const FewParams& p_in, hipStream_t stream) {
  FewParams p = p_in;
  p.tiles_m = (p.pixels + 16 * TM - 1) / (16 * TM);
  p.tiles_n = (p.oc + 16 * TN - 1) / (16 * TN);
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n)), block(64 * NW);
  hipLaunchKernelGGL((conv_few_kernel<T, TM, TN, NW, DEPTH>), grid, block, 0, stream, p);
  CINN_HIP_CALL(hipGetLastError());
}

// A tile's launch, in us: a block's start and end, what its CU pulls in (GB/s = 1e-3 KB/us) and multiplies, rounds of blocks
// beyond those that a CU holds.  Fitted to 330 layers of 1 to 32 images (0.14 in the logarithm, 2% from the best tile on average).
double Estimate(const FewParams& p, bool fp32, int tm, int tn, int nw, int depth) {
  const double blocks   = std::ceil(p.pixels / (16.0 * tm)) * std::ceil(p.oc / (16.0 * tn)), per_cu = std::ceil(blocks / 256);
  const int resident    = std::min(160 / (nw * depth * (tm + tn) * 2), 8);
  const double pulled   = per_cu * (tm + tn) * 2.048 * p.steps / 147;
  const double multiply = per_cu * p.steps * tm * tn * (fp32 ? 8 * 32 : 2 * 16) / 4 / 1938.0;
  return 3.0 + std::max(pulled, multiply) + 0.43 * std::min(pulled, multiply) + 1.15 * (std::ceil(per_cu / resident) - 1) + 0.043 * p.steps / nw;
}

template <typename T>
void Run(const FewParams& p, hipStream_t stream) {
  struct Tile {
    int tm, tn, nw, depth;
    void (*launch)(const FewParams&, hipStream_t);
  };
  // (four K steps in flight, or eight wavefronts for the larger tiles, leave room for one block on a CU: slower with
  // more blocks than CUs and no faster with fewer; 64x64 tiles lose to the tiled kernels wherever they beat the others)
  static const Tile tiles[] = {{1, 1, 8, 2, Launch<T, 1, 1, 8, 2>}, {1, 1, 4, 2, Launch<T, 1, 1, 4, 2>}, {1, 2, 4, 2, Launch<T, 1, 2, 4, 2>},
                               {2, 2, 4, 2, Launch<T, 2, 2, 4, 2>}, {2, 4, 4, 2, Launch<T, 2, 4, 4, 2>}};
  const Tile* best = nullptr;
  double best_us   = 0.0;
  for (const Tile& t : tiles) {
    const double us = Estimate(p, sizeof(T) == 4, t.tm, t.tn, t.nw, t.depth);
    if (!best || us < best_us) best = &t, best_us = us;
  }
  best->launch(p, stream);
}

}  // namespace

// FLAGS_cinn_hip_conv_few=0 switches the kernel off.
bool TryConvFew(const ConvNhwcArgs& a, hipStream_t stream) {
  static const bool enabled = !(getenv("FLAGS_cinn_hip_conv_few") && atoi(getenv("FLAGS_cinn_hip_conv_few")) == 0);
  if (!enabled || a.nchw_input || a.pool_after || a.x2) return false;
  const bool is_float = a.type.code == cinn_type_float && (a.type.bits == 32 || a.type.bits == 16);
  const bool is_bf16  = a.type.code == cinn_type_bfloat && a.type.bits == 16;
  if (!is_float && !is_bf16) return false;
  // A convolution in fp32 without a layer's scale stays with the tiled kernels: the K
  // that they split for it is what the tests of scratch memory under graph replay hold on to.
  if (a.type.bits == 32 && !a.scale) return false;
  // whole K steps inside a filter tap, whole groups of four channels of a result
  const int elem = a.type.bits / 8, lanes = kStepBytes / elem;
  if (a.c % lanes != 0 || a.oc % 4 != 0) return false;
  for (const void* ptr : {a.x, a.w, static_cast<const void*>(a.y), static_cast<const void*>(a.scale), static_cast<const void*>(a.shift), a.residual})
    if (reinterpret_cast<uintptr_t>(ptr) % 16 != 0) return false;
  // byte offsets are 32 bits wide, positions in the image are signed
  constexpr int64_t kLimit = (int64_t)1 << 31;
  const int64_t k_total = (int64_t)a.kh * a.kw * a.c, pixels = (int64_t)a.n * a.oh * a.ow;
  if ((int64_t)a.n * a.h * a.w_in * a.c * elem >= kLimit || a.oc * k_total * elem >= kLimit) return false;
  // Up to half as many tiles of 64x64 as CUs: beyond that the tiled kernels' larger tiles pull in less.  us, tiled | here: 98 tiles
  // (fp16, 256 -> 256 3x3 on 14x14, 8 images) 10.9 | 8.4, 104 (fp32, 512 -> 512 3x3 on 7x7, 16 images) 52.0 | 44.2, 112 (512 -> 1024 1x1 on
  // 14x14, 2 images) 6.1 | 5.1; 154 (192 -> 40 7x7) 28.8 | 33.2, 180 (960 -> 332 3x3) 34.0 | 36.7, 196 (256 -> 128 1x1 on 56x56, 2 images) 4.6 | 6.2.
  if (((pixels + 63) / 64) * ((a.oc + 63) / 64) > 128 || pixels < 1) return false;
  // (a single K step of few rows has nothing to share: 1 x 64 -> 4096 2.4 | 3.0, 8 x 64 -> 4096 2.9 | 3.0; 3136 x 64 -> 64 and more gain)
  if (k_total == lanes && pixels <= 16) return false;
  const bool outside = a.pad_h > 0 || a.pad_w > 0 || (int64_t)(a.oh - 1) * a.stride_h - a.pad_h + (int64_t)(a.kh - 1) * a.dil_h >= a.h ||
                       (int64_t)(a.ow - 1) * a.stride_w - a.pad_w + (int64_t)(a.kw - 1) * a.dil_w >= a.w_in;
  if (outside && !HasZeroPage(stream)) return false;
  FewParams p{};
  p.x = a.x, p.w = a.w, p.y = a.y, p.scale = a.scale, p.shift = a.shift, p.residual = a.residual;
  p.zeros = outside ? ConvZeroPage() : nullptr;
  p.h = a.h, p.w_in = a.w_in, p.c = a.c, p.oc = a.oc, p.pixels = (int)pixels, p.kw = a.kw;
  p.pad_h = a.pad_h, p.pad_w = a.pad_w, p.stride_h = a.stride_h, p.stride_w = a.stride_w, p.dil_h = a.dil_h, p.dil_w = a.dil_w;
  p.steps         = (int)(k_total * elem / kStepBytes);
  p.steps_per_tap = a.c / lanes;
  p.oh_ow = a.oh * a.ow, p.ow = a.ow;
  MagicFor(p.oh_ow, &p.magic_plane, &p.shift_plane);
  MagicFor(p.ow, &p.magic_ow, &p.shift_ow);
  p.relu = a.relu, p.alpha = a.alpha, p.residual_scale = a.residual_scale;
  // the larger operand is read from memory once: its rows go to one XCD
  p.pixels_outer = (int64_t)a.n * a.h * a.w_in * a.c > a.oc * k_total;
  if (is_bf16) {
    Run<__bf16>(p, stream);
  } else if (elem == 2) {
    Run<_Float16>(p, stream);
  } else {
    Run<float>(p, stream);
  }
  return true;
}

}  // namespace cinn_hip_kernels
