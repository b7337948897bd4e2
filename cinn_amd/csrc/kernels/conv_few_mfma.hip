// Channels-last convolutions of few output tiles for gfx950: one image, or a few, through a network's deeper stages; and layers
// of few filters, whose tiles of 64 columns would be mostly padding.
//
//   y[pixel][oc] = act( sum_k im2col(x)[pixel][k] w[oc][k] * scale + shift + residual ),  fp16 / bf16 / fp32
//
// The tiled kernels give such a layer 26 to 104 blocks of 64x64, split K over more blocks and add the parts in a second
// launch.  What bounds it is none of the chip's rates but one block's chain: launch, first operands, K steps with a block
// barrier each, partial sums to memory, launch, partial sums back.  Here the wavefronts of a block split K among themselves
// (few_tile.h), so that a layer is one launch of small output tiles, a block for most CUs.
//
// What bounds it then is what one CU pulls in: with fragments loaded straight into registers, in an order of lanes that
// pulls in a third as much, the same kernel took 6.55 us for 256 -> 256 3x3 on 14x14.  us, tiled kernels | here, fp16, one
// image, weights in the last-level cache: 128 -> 128 3x3 on 28x28 9.2 | 3.8, 256 -> 256 3x3 on 14x14 9.6 | 4.1, 1024 -> 256 1x1 7.6 | 3.4,
// 512 -> 512 3x3 on 7x7 10.5 | 5.2; fp32 15.1 | 6.5, 12.3 | 4.6, 20.9 | 9.7.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstdlib>

#include "kernels/conv_nhwc.h"
#include "kernels/few_tile.h"
#include "kernels/launch_count.h"
#include "runtime/hip_check.h"
#include "runtime/scratch.h"

namespace cinn_hip_kernels {

std::atomic<long long> g_launches[kCounted];

namespace {

using few::f32x4;

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

// TM x TN fragments of 16 pixels x 16 channels, NW wavefronts that share K.
template <typename T, int TM, int TN, int NW>
__global__ void __launch_bounds__(64 * NW)
conv_few_kernel(FewParams p) {
  typedef few::Ring<T, TM, TN> Ring;
  constexpr int E = (int)sizeof(T);
  __shared__ __attribute__((aligned(1024))) char lds[NW * Ring::BYTES];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Ring ring(lds, wave, lane);
  int tm, tn;
  few::TileOf(blockIdx.x, p.tiles_m, p.tiles_n, p.pixels_outer, &tm, &tn);
  const int m0 = tm * (16 * TM), n0 = tn * (16 * TN);
  int y0[2 * TM], x0[2 * TM];  // top left corner of the lane's pixels' windows
  unsigned off[2 * TM];        // byte offset of the lane's chunk there, modulo 2^32
  unsigned w_off[2 * TN];
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i) {
    const int row   = 8 * (i & 1) + (lane >> 3);
    const int chunk = few::ChunkAt(lane & 7, row) << 4;
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
    const int chunk = few::ChunkAt(lane & 7, row) << 4;
    w_off[j]        = (unsigned)min(n0 + 8 * j + (lane >> 3), p.oc - 1) * (unsigned)(p.steps * few::kStepBytes) + chunk;
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
#pragma unroll
    for (int j = 0; j < 2 * TN; ++j)
      few::CopyAt(ring.W(slot, j), static_cast<const char*>(p.w) + (int64_t)next * few::kStepBytes, w_off[j]);
    const unsigned tap_at = (unsigned)((dy * p.dil_h) * p.w_in + dx * p.dil_w) * (unsigned)(p.c * E) + (unsigned)(in_tap * few::kStepBytes);
#pragma unroll
    for (int i = 0; i < 2 * TM; ++i) {
      const bool inside = (unsigned)(y0[i] + dy * p.dil_h) < (unsigned)p.h && (unsigned)(x0[i] + dx * p.dil_w) < (unsigned)p.w_in;
      few::CopyAt(ring.X(slot, i), inside ? static_cast<const char*>(p.x) + (off[i] + tap_at) : static_cast<const char*>(p.zeros) + ((lane & 7) << 4));
    }
    if (++in_tap == p.steps_per_tap) {
      in_tap = 0;
      if (++dx == p.kw) dx = 0, ++dy;
    }
    ++next;
  };
  ring.Run(s1 - s0, request);
  ring.template Meet<NW>(lds, wave, lane, [&](int f, int i, int j, f32x4 sum) {
    const int pixel = m0 + 16 * i + (lane & 15), col = n0 + 16 * j + (lane >> 4) * 4;
    if (pixel >= p.pixels || col >= p.oc) return;
    vec4 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = __builtin_fmaf(sum[e], sc[f][e], sh[f][e]);
      if (p.residual) v = __builtin_fmaf(p.residual_scale, (float)res[f][e], v);
      asm volatile("" : "+v"(v));  // fp32 first, then one rounding to T
      out[e] = (T)(p.relu ? fmaxf(v, 0.0f) : v);
    }
    *reinterpret_cast<vec4*>(static_cast<T*>(p.y) + (int64_t)pixel * p.oc + col) = out;
  });
}

// q = (n * magic) >> shift == n / d for 0 <= n < 2^31
void MagicFor(int d, unsigned* magic, unsigned* shift) {
  int l = 0;
  while ((1ll << l) < d) ++l;
  *shift = d == 1 ? 0 : 31 + l;
  *magic = d == 1 ? 1 : (unsigned)(((1ull << *shift) / (unsigned)d) + 1);
}

template <typename T, int TM, int TN, int NW>
void Launch(const FewParams& p_in, hipStream_t stream) {
  FewParams p = p_in;
  p.tiles_m = (p.pixels + 16 * TM - 1) / (16 * TM);
  p.tiles_n = (p.oc + 16 * TN - 1) / (16 * TN);
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n)), block(64 * NW);
  hipLaunchKernelGGL((conv_few_kernel<T, TM, TN, NW>), grid, block, 0, stream, p);
  CINN_HIP_CALL(hipGetLastError());
}

struct Tile {
  int tm, tn, nw;
};
// (four K steps in flight, or eight wavefronts for the larger tiles, leave room for one block on a CU: slower with
// more blocks than CUs and no faster with fewer; 64x64 tiles lose to the tiled kernels wherever they beat the others)
constexpr Tile kTiles[] = {{1, 1, 8}, {1, 1, 4}, {1, 2, 4}, {2, 2, 4}, {2, 4, 4}};

// index of the fastest tile, and its estimate
int Choose(const FewParams& p, bool fp32, double* us) {
  int best = 0;
  for (int i = 0; i < (int)(sizeof(kTiles) / sizeof(Tile)); ++i) {
    const double t = few::Estimate(p.pixels, p.oc, p.steps, fp32, kTiles[i].tm, kTiles[i].tn, kTiles[i].nw);
    if (i == 0 || t < *us) best = i, *us = t;
  }
  return best;
}

template <typename T>
void Run(const FewParams& p, int tile, hipStream_t stream) {
  CountLaunch(kCountConvFew + tile);
  switch (tile) {
    case 0: Launch<T, 1, 1, 8>(p, stream); break;
    case 1: Launch<T, 1, 1, 4>(p, stream); break;
    case 2: Launch<T, 1, 2, 4>(p, stream); break;
    case 3: Launch<T, 2, 2, 4>(p, stream); break;
    default: Launch<T, 2, 4, 4>(p, stream); break;
  }
}

// us of the tiled kernels; fitted to 140 layers in fp32, 1x1 to 7x7 (9% off on average), and 62 of more than 128 tiles in 16 bits (17%;
// 105 of up to 128 tiles: 10%)
double TiledMicroseconds(const FewParams& p, bool fp32) {
  const int tiles  = (int)std::min<int64_t>((int64_t)((p.pixels + 63) / 64) * ((p.oc + 63) / 64), 1 << 24);
  const int splits = ConvSplits(tiles, p.steps, fp32), share = (p.steps + splits - 1) / splits;
  const double cus = (double)tiles * splits / 256, mb = (double)p.pixels * p.oc * (fp32 ? 4e-6 : 2e-6);
  if (fp32) {
    const double per_cu = tiles < 256 ? std::ceil(cus) : cus;
    return 4.0 + (per_cu <= 1.0 ? 0.65 : 0.6 * per_cu) * share + 0.4 * mb + (splits > 1 ? 2.4 + 0.25 * splits * mb : 0.0);
  }
  return 4.45 + 0.266 * std::max(cus, 1.0) * share + 0.14 * mb + (splits > 1 ? 3.7 + 0.39 * splits * mb : 0.0);
}

}  // namespace

namespace {

// 1: by the rules below (default), 0: never; -1: not read yet
std::atomic<int> g_few_mode{-1};

int FewMode() {
  int mode = g_few_mode.load(std::memory_order_relaxed);
  if (mode < 0) {
    const char* v = getenv("FLAGS_cinn_hip_conv_few");
    mode          = v && *v ? (atoi(v) != 0) : 1;
    g_few_mode.store(mode, std::memory_order_relaxed);
  }
  return mode;
}

// TryProductFew, and TryConvFew with limit_us < 0
double TryFew(const ConvNhwcArgs& a, double limit_us, bool dry, hipStream_t stream) {
  if (FewMode() == 0 || a.nchw_input || a.pool_after || a.x2) return 0.0;
  const bool is_float = a.type.code == cinn_type_float && (a.type.bits == 32 || a.type.bits == 16);
  const bool is_bf16  = a.type.code == cinn_type_bfloat && a.type.bits == 16;
  if (!is_float && !is_bf16) return 0.0;
  // whole K steps inside a filter tap, whole groups of four channels of a result
  const int elem = a.type.bits / 8, lanes = few::kStepBytes / elem;
  if (a.c % lanes != 0 || a.oc % 4 != 0) return 0.0;
  for (const void* ptr : {a.x, a.w, static_cast<const void*>(a.y), static_cast<const void*>(a.scale), static_cast<const void*>(a.shift), a.residual})
    if (reinterpret_cast<uintptr_t>(ptr) % 16 != 0) return 0.0;
  // byte offsets are 32 bits wide, positions in the image are signed
  constexpr int64_t kLimit = (int64_t)1 << 31;
  const int64_t k_total = (int64_t)a.kh * a.kw * a.c, pixels = (int64_t)a.n * a.oh * a.ow;
  if ((int64_t)a.n * a.h * a.w_in * a.c * elem >= kLimit || a.oc * k_total * elem >= kLimit) return 0.0;
  // (512 threads for each tile of 16x16: fewer than 2^32 of a launch)
  if (pixels < 1 || pixels >= (1 << 24) || pixels * a.oc >= (1 << 30)) return 0.0;
  // A convolution goes by the two estimates.  Up to half as many tiles of 64x64 as CUs most are far apart: us, tiled | here, in fp16
  // 98 tiles (256 -> 256 3x3 on 14x14, 8 images) 14.0 | 7.9, in fp32 26 tiles (128 -> 128 3x3 on 28x28) 13.0 | 6.7, 49 (64 -> 64 3x3 on 56x56) 11.7 | 6.6.
  // What is even or slower is a long K, shared by four or eight wavefronts instead of up to eight blocks of four.  In 16 bits, 105 layers of up
  // to 128 tiles: below 0.97 of the tiled kernels' estimate 93 of 94 are faster or even (0.99 to 2.4; 320 -> 448 7x7 on 29x32 27.2 | 29.8 is the
  // other one), above it 9 of 11 slower or even (512 -> 144 7x7 on 39x49 40.3 | 46.2).  In fp32, 70 layers: of less than 200 steps below 0.95 44 are 0.97 to 2.6
  // times as fast, above it 6 0.86 to 1.02 (448 -> 64 3x3 on 45x28, 5 images, 39.6 | 45.5); of more below 0.9 5 1.05 to 1.2, above it 15 0.73 to 1.0 (384 ->
  // 64 7x7 on 57x57 82.8 | 112.9).  The filters' scale has no part in it.
  // Beyond, the tiled kernels' larger tiles pull in less, but a tile's columns are 64: layers of 8 to 60 filters, or a few more than
  // a multiple of 64, multiply mostly padding there.  60 layers in fp16 of 132 to 1168
  // tiles: 23 are a fifth below, 1.17 to 2.3 times faster (64 -> 16 7x7 on 38x22, 24 images, 25.1 | 11.4; 512 -> 12 5x5 on 57x56, 3 images, 16.3 | 7.8), none slower;
  // of the others 316 tiles (384 -> 72 5x5) 33.3 | 43.9, 485 (256 -> 304 1x1) 6.3 | 11.2, 945 (128 -> 192 3x3) 22.6 | 34.4.  A multiple of 64 has no
  // such columns: 196 tiles (256 -> 128 1x1 on 56x56, 2 images) 4.6 | 6.2.
  // In fp32 these tiles are bound by the matrix pipe, and whole columns gain as well, but four steps and fewer are bound by what they
  // store: 1 (32 -> 384 1x1 on 43x30, 2 images) 4.9 | 7.9, 3 (96 -> 192 1x1 on 14x46, 8 images) 6.5 | 8.2, 4 (128 -> 40 1x1 / 2) 6.5 | 6.7.  From 5 steps
  // on a fifth below: 140 layers 1.16 to 3.8 times faster (480 -> 16 1x1 / 2 on 16x11, 27 images, 12.9 | 3.4), 37 of 129 to 426 tiles 0.97 to 1.8
  // (64 -> 512 3x3 / 2 on 37x24, 5 images, 16.1 | 13.5); of those not taken 404 tiles (256 -> 128 1x1) 14.4 | 16.6, 836 (32 -> 256 3x3 / 2) 26.0 | 42.9.
  const bool few_tiles = ((pixels + 63) / 64) * ((a.oc + 63) / 64) <= 128;
  if (limit_us < 0.0 && !few_tiles && (elem == 2 ? a.oc % 64 == 0 : k_total <= 4 * lanes)) return 0.0;
  // (a single K step of few rows has nothing to share: 1 x 64 -> 4096 2.4 | 3.0, 8 x 64 -> 4096 2.9 | 3.0; 3136 x 64 -> 64 and more gain)
  if (k_total == lanes && pixels <= 16) return 0.0;
  const bool outside = a.pad_h > 0 || a.pad_w > 0 || (int64_t)(a.oh - 1) * a.stride_h - a.pad_h + (int64_t)(a.kh - 1) * a.dil_h >= a.h ||
                       (int64_t)(a.ow - 1) * a.stride_w - a.pad_w + (int64_t)(a.kw - 1) * a.dil_w >= a.w_in;
  if (outside && !HasZeroPage(stream)) return 0.0;
  FewParams p{};
  p.x = a.x, p.w = a.w, p.y = a.y, p.scale = a.scale, p.shift = a.shift, p.residual = a.residual;
  p.zeros = outside ? ConvZeroPage() : nullptr;
  p.h = a.h, p.w_in = a.w_in, p.c = a.c, p.oc = a.oc, p.pixels = (int)pixels, p.kw = a.kw;
  p.pad_h = a.pad_h, p.pad_w = a.pad_w, p.stride_h = a.stride_h, p.stride_w = a.stride_w, p.dil_h = a.dil_h, p.dil_w = a.dil_w;
  p.steps         = (int)(k_total * elem / few::kStepBytes);
  p.steps_per_tap = a.c / lanes;
  p.oh_ow = a.oh * a.ow, p.ow = a.ow;
  MagicFor(p.oh_ow, &p.magic_plane, &p.shift_plane);
  MagicFor(p.ow, &p.magic_ow, &p.shift_ow);
  p.relu = a.relu, p.alpha = a.alpha, p.residual_scale = a.residual_scale;
  // the larger operand is read from memory once: its rows go to one XCD
  p.pixels_outer = (int64_t)a.n * a.h * a.w_in * a.c > a.oc * k_total;
  double us;
  const int tile = Choose(p, elem == 4, &us);
  const double share = !few_tiles ? 0.8 : elem == 2 ? 0.97 : p.steps < 200 ? 0.95 : 0.9;
  if (us >= (limit_us < 0.0 ? share * TiledMicroseconds(p, elem == 4) : limit_us)) return 0.0;
  if (dry) return us;
  if (is_bf16) {
    Run<__bf16>(p, tile, stream);
  } else if (elem == 2) {
    Run<_Float16>(p, tile, stream);
  } else {
    Run<float>(p, tile, stream);
  }
  return us;
}

}  // namespace

bool TryConvFew(const ConvNhwcArgs& a, hipStream_t stream) { return TryFew(a, -1.0, false, stream) > 0.0; }

double TryProductFew(const ConvNhwcArgs& a, double limit_us, bool dry, hipStream_t stream) { return TryFew(a, limit_us, dry, stream); }

}  // namespace cinn_hip_kernels

// FLAGS_cinn_hip_conv_few=0, or a mode of 0, switches the kernel off.
extern "C" int cinn_hip_conv_few_mode(int mode) {
  const int before = cinn_hip_kernels::FewMode();
  if (mode == 0 || mode == 1) cinn_hip_kernels::g_few_mode.store(mode, std::memory_order_relaxed);
  return before;
}

extern "C" long long cinn_hip_launches(int which) {
  return which >= 0 && which < cinn_hip_kernels::kCounted ? cinn_hip_kernels::g_launches[which].load(std::memory_order_relaxed) : -1;
}
