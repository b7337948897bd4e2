// Gradients of a convolution on the MFMA units (gfx950), fp16 / bf16 / fp32, channels last inside.
//
// Both gradients are matrix products over tensors whose channels are contiguous:
//   dx[pixel][c]      = sum over (tap, f)  dy[pixel - tap][f] * w[f][tap][c]
//   dw[f][(tap, c)]   = sum over pixels    dy[pixel][f] * x[pixel + tap][c]
//
//   * dx at stride 1 is a forward convolution of dy with the filter turned round, [c][tap'][f]: it runs on the forward
//     kernels (RunConvNhwc) after one small kernel has rearranged the filter.
//   * dx at a larger stride: the input pixels of one remainder class (iy mod stride, ix mod stride) see the same taps,
//     every stride-th one, and neighbouring pixels of the class see neighbouring dy.  Each class is a product of its own
//     (pixels x channels, K = its taps x f), all classes in one launch; no multiply-add meets an inserted zero.
//     Taps outside dy meet a zero in either form, as in the forward convolution: an infinite filter value makes NaN there.
//     (A kernel that computes such pixels again would be one more launch, 2.8 us of the 16 that a 64 -> 64 3x3 layer on
//     56x56 at batch 32 takes in fp16; whoever has such a filter has the NaNs from the forward pass.)
//   * dw: rows are filters, columns (tap, channel), and K runs over all output pixels, which both operands keep as their
//     slow axis: they lie in LDS as [pixel][channels] and are read with transposing reads.  The x operand is gathered
//     row by row (a chunk of channels of pixel + tap, or zeros); at a stride of one the taps of a filter row share what is
//     read (conv_filter_taps_kernel).  K is long (1e5) and the result small, so K is split until the chip is full; the
//     fp32 planes are added by a second kernel, which also writes the filter's own layout.
// Measured before (one thread or block per gradient element) and here: 64 -> 64 3x3 on 56x56 at batch 32 in fp16, NCHW,
// dx 4988 -> 13 us (560 TFLOP/s) and dw 9467 -> 28 + 6 us (with the x operand read nine times from L2), 19 + 5 us by
// neighbouring taps, with 5 to 7 us for each copied tensor; 96 -> 200 3x3 / stride 2 on 35x41 at batch 8 in fp32, dx 1661 -> 31 us and dw
// 3844 -> 22 + 5 us (47 TFLOP/s).
// Tensors that are not channels last, or whose channel count is no multiple of a 16-byte chunk, are first copied into
// that form in scratch (pack_kernel), and dx is copied back (with beta, after it has been copied there).
#include "kernels/conv_backward.h"

#include <algorithm>
#include <climits>

#include "kernels/conv_nhwc.h"
#include "kernels/flex_tile.h"
#include "runtime/hip_check.h"
#include "runtime/scratch.h"

namespace cinn_hip_kernels {
namespace {

using flex::u32x4;

// ---- copies between tensor layouts ---------------------------------------------------------------------------------
// [n][c][plane] (nchw) or [n][plane][c] -> [n][plane][cp], channels c .. cp-1 zero.  A block moves 64 pixels x 64
// channels of one image through LDS.
template <typename T, bool NCHW>
__global__ void __launch_bounds__(256)
pack_kernel(const T* __restrict__ in, T* __restrict__ out, int c, int plane, int cp) {
  constexpr int E = 16 / (int)sizeof(T), CPR = 64 / E;  // chunks per 64-element row
  __shared__ T tile[64][64 + 4 / (int)sizeof(T)];       // [pixel][channel]
  const int p0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
  in += (int64_t)blockIdx.z * c * plane;
  out += (int64_t)blockIdx.z * plane * cp;
  const int rows = NCHW ? c : plane, cols = NCHW ? plane : c;  // memory is [rows][cols]
  const int r0 = NCHW ? c0 : p0, q0 = NCHW ? p0 : c0;
  for (int u = threadIdx.x; u < 64 * CPR; u += 256) {
    const int r = u / CPR, q = u % CPR * E;
    typedef T chunk_t __attribute__((ext_vector_type(E)));
    chunk_t v = {0};
    if (r0 + r < rows) {
      const T* from = in + (int64_t)(r0 + r) * cols + q0 + q;
      if (q0 + q + E <= cols) {
        __builtin_memcpy(&v, from, 16);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e)
          if (q0 + q + e < cols) v[e] = from[e];
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) (NCHW ? tile[q + e][r] : tile[r][q + e]) = v[e];
  }
  __syncthreads();
  for (int u = threadIdx.x; u < 64 * CPR; u += 256) {
    const int p = u / CPR, q = u % CPR * E;
    if (p0 + p >= plane || c0 + q >= cp) continue;
    T v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = tile[p][q + e];
    T* to = out + (int64_t)(p0 + p) * cp + c0 + q;
    if (c0 + q + E <= cp) {
      __builtin_memcpy(to, v, 16);
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (c0 + q + e < cp) to[e] = v[e];
    }
  }
}

// [n][plane][c] -> [n][c][plane]
template <typename T>
__global__ void __launch_bounds__(256)
unpack_kernel(const T* __restrict__ in, T* __restrict__ out, int c, int plane) {
  constexpr int E = 16 / (int)sizeof(T), CPR = 64 / E;
  __shared__ T tile[64][64 + 4 / (int)sizeof(T)];  // [pixel][channel]
  const int p0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
  in += (int64_t)blockIdx.z * c * plane;
  out += (int64_t)blockIdx.z * plane * c;
  for (int u = threadIdx.x; u < 64 * CPR; u += 256) {
    const int p = u / CPR, q = u % CPR * E;
    typedef T chunk_t __attribute__((ext_vector_type(E)));
    chunk_t v = {0};
    if (p0 + p < plane) {
      const T* from = in + (int64_t)(p0 + p) * c + c0 + q;
      if (c0 + q + E <= c) {
        __builtin_memcpy(&v, from, 16);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e)
          if (c0 + q + e < c) v[e] = from[e];
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) tile[p][q + e] = v[e];
  }
  __syncthreads();
  for (int u = threadIdx.x; u < 64 * CPR; u += 256) {
    const int r = u / CPR, q = u % CPR * E;  // channel, first pixel
    if (c0 + r >= c) continue;
    T* to = out + (int64_t)(c0 + r) * plane + p0 + q;
    typedef T chunk_t __attribute__((ext_vector_type(E)));
    chunk_t v;
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = tile[q + e][r];
    if (p0 + q + E <= plane) {
      __builtin_memcpy(to, &v, 16);
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (p0 + q + e < plane) to[e] = v[e];
    }
  }
}

// The filter as the data gradient reads it: a slot for every first tap (ky0, kx0) of a class, i.e. for every class that has
// taps at all (whatever the stride, slots do not add up to more than the filter with its extents rounded up), then
// [c][i][j][fp] with i, j counting the class's taps ky = ky0 + stride i, kx likewise; f .. fp-1 are zero.  Stride 1 (one
// class): the forward kernel walks the taps upwards in dy, so they are turned round.
struct FilterParams {
  int f, c, kh, kw, fp;
  int nhwc;                    // filter [f][kh][kw][c], else [f][c][kh][kw]
  int stride_h, stride_w;
  int slots_w;                 // slots side by side: first taps kx0
  int turn;                    // 1: turned round (stride 1)
  int64_t slot;                // elements of a slot
};
template <typename T>
__global__ void __launch_bounds__(256)
filter_kernel(const T* __restrict__ w, T* __restrict__ out, FilterParams p) {
  const int ky0 = blockIdx.y / p.slots_w, kx0 = blockIdx.y % p.slots_w;  // below the stride and the extent
  const int nky = (p.kh - 1 - ky0) / p.stride_h + 1, nkx = (p.kw - 1 - kx0) / p.stride_w + 1;
  const int64_t total = (int64_t)p.c * nky * nkx * p.fp;
  const int64_t idx   = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= total) return;
  const int f = (int)(idx % p.fp);
  int rest    = (int)(idx / p.fp);
  const int j = rest % nkx;
  rest /= nkx;
  const int i = rest % nky, c = rest / nky;
  const int ky = p.turn ? p.kh - 1 - i : ky0 + p.stride_h * i;
  const int kx = p.turn ? p.kw - 1 - j : kx0 + p.stride_w * j;
  T v = (T)0.0f;
  if (f < p.f)
    v = p.nhwc ? w[(((int64_t)f * p.kh + ky) * p.kw + kx) * p.c + c] : w[(((int64_t)f * p.c + c) * p.kh + ky) * p.kw + kx];
  out[blockIdx.y * p.slot + idx] = v;
}

// ---- data gradient at a stride -------------------------------------------------------------------------------------
struct DataParams {
  const void* dy;    // [n][oh][ow][fp]
  const void* wt;    // class slots of filter_kernel
  void* dx;          // [n][h][w][c]
  const void* zeros;
  int n, h, w, c, oh, ow, fp, kh, kw;
  int stride_h, stride_w, pad_h, pad_w;
  int slots_w;
  int64_t slot;
  float alpha, beta;
};

// rows are the pixels of one remainder class, K = (tap i, tap j, f): a chunk is 16 bytes of dy's pixel
// (jy + oy0 - i, jx + ox0 - j), or zeros.  Load() is called for consecutive steps.
template <typename T, int ROWS, int THREADS>
struct DataTile {
  static constexpr int E = 16 / (int)sizeof(T), KS = 8 * E, CHUNKS = ROWS * 8 / THREADS;
  const T* dy;
  const T* zeros;
  int oh, ow, fp, nky, nkx;
  int base[CHUNKS], oy[CHUNKS], ox[CHUNKS];
  int f, i, j;  // position of the thread's chunk in the reduction

  __device__ __forceinline__ void Init(const DataParams& p, int row0, int rows, int hc, int wc, int oy0, int ox0, int nky_, int nkx_,
                                       int tid) {
    dy = static_cast<const T*>(p.dy), zeros = static_cast<const T*>(p.zeros);
    oh = p.oh, ow = p.ow, fp = p.fp, nky = nky_, nkx = nkx_;
#pragma unroll
    for (int q = 0; q < CHUNKS; ++q) {
      const int m  = min(row0 + (tid >> 3) + THREADS / 8 * q, rows - 1);
      const int jx = m % wc, jy = m / wc % hc, n = m / (wc * hc);
      oy[q] = jy + oy0, ox[q] = jx + ox0;
      base[q] = ((n * oh + oy[q]) * ow + ox[q]) * fp;
    }
    f = (tid & 7) * E;
    i = j = 0;
    Wrap();
  }
  __device__ __forceinline__ void Wrap() {
    while (f >= fp) {
      f -= fp;
      if (++j >= nkx) j = 0, ++i;
    }
  }
  template <bool GUARD>
  __device__ __forceinline__ void Load(u32x4 (&r)[CHUNKS], int, int, int) {
    const int tap = f - (i * ow + j) * fp;
#pragma unroll
    for (int q = 0; q < CHUNKS; ++q) {
      const bool ok = i < nky && (unsigned)(oy[q] - i) < (unsigned)oh && (unsigned)(ox[q] - j) < (unsigned)ow;
      r[q] = *reinterpret_cast<const u32x4*>(ok ? dy + (base[q] + tap) : zeros);
    }
    f += KS;
    Wrap();
  }
  __device__ __forceinline__ void Store(char* tile, const u32x4 (&r)[CHUNKS], int tid) const {
#pragma unroll
    for (int q = 0; q < CHUNKS; ++q)
      *reinterpret_cast<u32x4*>(tile + flex::Tile<T, true, ROWS, THREADS>::LdsOffset(tid, q)) = r[q];
  }
};

template <typename T, int BM, int BN>
__global__ void __launch_bounds__(256, 2)
conv_data_kernel(DataParams p) {
  __shared__ __attribute__((aligned(256))) char lds[2 * (BM + BN) * 128];
  constexpr int KS = 128 / (int)sizeof(T);
  const int tid = threadIdx.x;
  const int ry = blockIdx.y / p.stride_w, rx = blockIdx.y % p.stride_w;
  const int hc = (p.h - ry + p.stride_h - 1) / p.stride_h, wc = (p.w - rx + p.stride_w - 1) / p.stride_w;
  const int rows = hc > 0 && wc > 0 ? p.n * hc * wc : 0;
  const int ky0 = (ry + p.pad_h) % p.stride_h, kx0 = (rx + p.pad_w) % p.stride_w;
  const int nky = ky0 < p.kh ? (p.kh - 1 - ky0) / p.stride_h + 1 : 0;
  const int nkx = kx0 < p.kw ? (p.kw - 1 - kx0) / p.stride_w + 1 : 0;
  const int k   = nky * nkx * p.fp;
  const int tiles_m = (rows + BM - 1) / BM, tiles_n = (p.c + BN - 1) / BN;
  if ((int)blockIdx.x >= tiles_m * tiles_n) return;  // the grid is the largest class's
  int tm, tn;
  flex::TileOf(blockIdx.x, tiles_m, tiles_n, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN;

  DataTile<T, BM, 256> ta;
  flex::Tile<T, true, BN, 256> tb;
  ta.Init(p, m0, rows, hc, wc, (ry + p.pad_h - ky0) / p.stride_h, (rx + p.pad_w - kx0) / p.stride_w, nky, nkx, tid);
  tb.Init(static_cast<const T*>(p.wt) + (k > 0 ? (ky0 * p.slots_w + kx0) * p.slot : 0), k, n0, p.c, k, tid);
  typename flex::Mma<T, true, true, BM, BN>::acc_t acc;
  flex::KLoop<T, true, true, BM, BN, 1>(lds, ta, tb, 0, (k + KS - 1) / KS, k / KS, k, tid, acc);

  const int col0 = n0 + tid % (BN / 8) * 8;
  const int cols = min(p.c - col0, 8);
  T* dx = static_cast<T*>(p.dx);
  flex::EachRowGroup<T, true, true, BM, BN, 1>(lds, acc, tid, [&](int row, int, const float (&v)[8]) {
    const int m = m0 + row;
    if (m >= rows || cols <= 0) return;
    const int jx = m % wc, jy = m / wc % hc, n = m / (wc * hc);
    T* to = dx + ((int64_t)(n * p.h + jy * p.stride_h + ry) * p.w + jx * p.stride_w + rx) * p.c + col0;
    typedef T vec8 __attribute__((ext_vector_type(8)));
    if (cols == 8) {
      vec8 out, old = {0, 0, 0, 0, 0, 0, 0, 0};
      if (p.beta != 0.0f) __builtin_memcpy(&old, to, 8 * sizeof(T));
#pragma unroll
      for (int e = 0; e < 8; ++e) out[e] = (T)__builtin_fmaf(p.beta, (float)old[e], p.alpha * v[e]);
      __builtin_memcpy(to, &out, 8 * sizeof(T));
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e < cols) to[e] = (T)__builtin_fmaf(p.beta, p.beta != 0.0f ? (float)to[e] : 0.0f, p.alpha * v[e]);
    }
  });
}

// ---- filter gradient -----------------------------------------------------------------------------------------------
struct FilterGradParams {
  const void* dy;   // [pixels][fp]
  const void* x;    // [n][h][w][cp]
  const void* zeros;
  float* planes;    // [split][f][kh kw cp]
  int f, fp, cp, h, w, oh, ow, kw, taps;
  int stride_h, stride_w, pad_h, pad_w, dil_h, dil_w;
  int pixels, steps, steps_per_split;
  int tiles_m, tiles_n;
  int adv_n, adv_oy, adv_ox;  // a K step in images, rows and columns of the output
  int spill;  // 1: taps meet zeros of dy inside the image too (conv_filter_taps_kernel)
};

// the x operand: [pixel][ROWS columns of (tap, channel)].  A thread's chunks share one column chunk, i.e. one tap;
// their pixels advance by one K step from call to call, carried through (ox, oy, n) without a division.
template <typename T, int ROWS, int THREADS>
struct ImageTile {
  typedef flex::Tile<T, false, ROWS, THREADS> Plain;
  static constexpr int E = Plain::E, KS = Plain::KS, CHUNKS = Plain::CHUNKS;
  const T* x;
  const T* zeros;
  int h, w, cp, oh, ow, stride_h, stride_w, adv_n, adv_oy, adv_ox, pixels;
  int dy, dx, c;  // the tap's offset and the first channel
  int image[CHUNKS], oy[CHUNKS], ox[CHUNKS];  // image: offset of the pixel's image, in pixels of x

  __device__ __forceinline__ void Init(const FilterGradParams& p, int col0, int step0, int tid) {
    x = static_cast<const T*>(p.x), zeros = static_cast<const T*>(p.zeros);
    h = p.h, w = p.w, cp = p.cp, oh = p.oh, ow = p.ow, stride_h = p.stride_h, stride_w = p.stride_w;
    adv_n = p.adv_n * h * w, adv_oy = p.adv_oy, adv_ox = p.adv_ox, pixels = p.pixels;
    const int col = min(col0 + tid % Plain::CH * E, p.taps * cp - E);  // what lies beyond the last column is not stored
    const int tap = col / cp;
    c  = col - tap * cp;
    dy = tap / p.kw * p.dil_h - p.pad_h;
    dx = tap % p.kw * p.dil_w - p.pad_w;
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      const int pixel = step0 * KS + Plain::ChunkK(tid, i);
      const int n     = pixel / (oh * ow), rest = pixel - n * (oh * ow);
      oy[i] = rest / ow, ox[i] = rest - oy[i] * ow;
      image[i] = n * h * w;
    }
  }
  template <bool GUARD>
  __device__ __forceinline__ void Load(u32x4 (&r)[CHUNKS], int step, int, int tid) {
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      const int iy = oy[i] * stride_h + dy, ix = ox[i] * stride_w + dx;
      const bool ok = (unsigned)iy < (unsigned)h && (unsigned)ix < (unsigned)w && (!GUARD || step * KS + Plain::ChunkK(tid, i) < pixels);
      r[i] = *reinterpret_cast<const u32x4*>(ok ? x + ((image[i] + iy * w + ix) * cp + c) : zeros);
      ox[i] += adv_ox;
      const bool row = ox[i] >= ow;
      ox[i] -= row ? ow : 0;
      oy[i] += adv_oy + (row ? 1 : 0);
      const bool next = oy[i] >= oh;
      oy[i] -= next ? oh : 0;
      image[i] += adv_n + (next ? h * w : 0);
    }
  }
  __device__ __forceinline__ void Store(char* tile, const u32x4 (&r)[CHUNKS], int tid) const {
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) *reinterpret_cast<u32x4*>(tile + Plain::LdsOffset(tid, i)) = r[i];
  }
};

template <typename T, int BM, int BN>
__global__ void __launch_bounds__(256, 2)
conv_filter_kernel(FilterGradParams p) {
  __shared__ __attribute__((aligned(256))) char lds[2 * (BM + BN) * 128];
  constexpr int KS = 128 / (int)sizeof(T);
  const int tid = threadIdx.x;
  int tm, tn;
  flex::TileOf(blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int s0 = blockIdx.y * p.steps_per_split, s1 = min(s0 + p.steps_per_split, p.steps);

  flex::Tile<T, false, BM, 256> ta;
  ImageTile<T, BN, 256> tb;
  ta.Init(p.dy, p.fp, m0, p.fp, p.pixels, tid);
  tb.Init(p, n0, s0, tid);
  typename flex::Mma<T, false, false, BM, BN>::acc_t acc;
  // fp32: every K step in two parts.  The gather kernel's 256 threads added pixels / 256 products each and their sums in
  // pairs; as one chain per split the error against float64 was up to three times larger.  Relative 2-norm, gather | one
  // chain | a step | two parts: 784 pixels 0.85e-7 | 2.25e-7 | 1.19e-7 | 1.00e-7, 12544 pixels 1.46 | 2.41 | 1.46 | 1.31,
  // 25088 pixels 1.91 | 3.26 | 1.53 | 1.38.  96 -> 200 3x3 / stride 2 on 35x35 at batch 8: 24.6 -> 25.5 us.
  constexpr int PARTS = sizeof(T) == 4 ? 2 : 0;
  flex::KLoop<T, false, false, BM, BN, 1, PARTS>(lds, ta, tb, s0, s1, p.pixels / KS, p.pixels, tid, acc);

  const int columns = p.taps * p.cp;  // a multiple of a chunk, not of eight, in fp32
  const int col0    = n0 + tid % (BN / 8) * 8;
  float* plane      = p.planes + (int64_t)blockIdx.y * p.f * columns;
  flex::EachRowGroup<T, false, false, BM, BN, 1>(lds, acc, tid, [&](int row, int, const float (&v)[8]) {
    const int m = m0 + row;
    if (m >= p.f) return;
    float* to = plane + (int64_t)m * columns + col0;
    if (col0 + 4 <= columns) __builtin_memcpy(to, v, 16);
    if (col0 + 8 <= columns) __builtin_memcpy(to + 4, v + 4, 16);
  });
}

// ---- filter gradient, neighbouring taps of a row ----------------------------------------------------------------------
// At a stride of one the taps kx, kx + 1 and kx + 2 of a filter row multiply the same dy by the same pixels of x, one apart.
// conv_filter_kernel reads x once for each of them; here a block's columns are 64 channels x three such taps, and one tile of x
// serves all three: of the four k a transposing read brings, three reads hold the eight of every tap (tap kx starts kx later).
//
// K runs over positions: the pixels of an output row and kTaps - 1 more behind it, where dy is taken as zero, so that the
// pixel a tap reads is the position's own plus the tap, in the same row.  A K step is 64 positions of which the last
// kTaps - 1 only lend their pixels to the ones before them (dy zero once more); the next step begins with them.
// Positions, image rows and addresses advance without a division; what is outside comes back as zero from the buffer loads'
// range check.  Zeros of dy meet pixels of the image, so NaNs are computed again for every tap (filter_reduce_kernel).
//
// Eight wavefronts: two halves of each K step, added in LDS at the end (half the planes of two blocks), each 2 x 2 over filters
// and channels.
// 64 -> 64 3x3 on 56x56 at batch 32, fp16: 27.2 -> 18.9 us (392 TFLOP/s) and the reduction of the planes 6.1 -> 4.7; 82 MB
// come out of L2 instead of 188, and 21 steps per block (of one per CU) take about half of the time, the rest is the launch,
// the first operands and 12 MB of planes.
constexpr int kTaps = 3, kFresh = 64 - (kTaps - 1);  // positions of a K step that are its own

struct TapsParams {
  FilterGradParams g;
  int tiles_c, groups, tiles;  // tiles: m fastest, then channels, groups of taps, rows of the filter
  int splits, lanes_log2;      // splits: a multiple of 1 << lanes_log2
  int period, rows;            // positions of an output row; output rows of all images
  int adv_at, adv_row;         // a K step in positions and rows
  int adv_oy, adv_n;           // adv_row in output rows and images
};

template <typename T>
__global__ void __launch_bounds__(512, 1)
conv_filter_taps_kernel(TapsParams p) {
  constexpr int BM = 64, BN = 64;                                                // filters, channels
  constexpr int A_BYTES = BM * 128, B_ROWS = 68, STAGE = A_BYTES + B_ROWS * 128;  // reads reach four rows beyond the step
  constexpr int COLS = kTaps * BN, SLD = COLS + 4;
  constexpr int TM = 2, TN = 2, PF = 4;
  typedef flex::Tile<T, false, 64, 512> Tile;  // a chunk of either operand per thread and step
  typedef flex::Mma<T, false, false, BM, BN> M;
  typedef typename M::vec8 vec8;
  static_assert(64 * SLD * 4 >= 2 * STAGE, "the staging tile of the results covers the stages");
  __shared__ __attribute__((aligned(256))) char lds[64 * SLD * 4];
  const FilterGradParams& g = p.g;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;

  // every split's tiles on one XCD (blocks go to the 8 of them in turn), one after the other: they read the same pixels
  const int order = blockIdx.x >> p.lanes_log2;
  const int split = (order / p.tiles << p.lanes_log2) + (blockIdx.x & ((1 << p.lanes_log2) - 1));
  int tile        = order % p.tiles;
  const int m0    = tile % g.tiles_m * BM;
  tile /= g.tiles_m;
  const int c0 = tile % p.tiles_c * BN;
  tile /= p.tiles_c;
  const int kx0 = tile % p.groups * kTaps, ky = tile / p.groups;
  const int s0 = split * g.steps_per_split, s1 = min(s0 + g.steps_per_split, g.steps);

  const __amdgpu_buffer_rsrc_t dy_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(g.dy), 0, g.pixels * g.fp * (int)sizeof(T), 0x00020000);
  const __amdgpu_buffer_rsrc_t x_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(g.x), 0, p.rows / g.oh * g.h * g.w * g.cp * (int)sizeof(T), 0x00020000);
  constexpr unsigned kOutside = 0x80000000u;

  // The thread's chunk of either operand: its position in the output row, the row of all images and of its image, offsets of
  // the row's first pixel.  Channels beyond the last chunk repeat it (and are not stored).
  const int k   = Tile::ChunkK(tid, 0);
  const int t   = s0 * kFresh + k;
  int row = t / p.period, at = t - row * p.period;
  const int image0 = row / g.oh, iy_first = ky * g.dil_h - g.pad_h, iy_end = g.oh * g.stride_h + iy_first, shift = kx0 - g.pad_w;
  int iy = (row - image0 * g.oh) * g.stride_h + iy_first;
  const unsigned a_line = (unsigned)(g.ow * g.fp), b_line = (unsigned)(g.w * g.cp);
  unsigned a_row = (unsigned)row * a_line, b_row = ((unsigned)(image0 * g.h) + (unsigned)iy) * b_line;
  const unsigned a_col = (unsigned)min(m0 + tid % Tile::CH * 8, g.fp - 8), b_col = (unsigned)min(c0 + tid % Tile::CH * 8, g.cp - 8);
  const unsigned a_step = (unsigned)p.adv_row * a_line, b_step = (unsigned)(p.adv_n * g.h + p.adv_oy * g.stride_h) * b_line;
  const unsigned b_next = (unsigned)g.stride_h * b_line, b_image = (unsigned)(g.h - g.oh * g.stride_h) * b_line;

  u32x4 ra[PF], rb[PF];
  auto load = [&](int slot) {
    const int ix    = at + shift;
    const bool a_ok = k < kFresh && at < g.ow && row < p.rows;
    const bool b_ok = (unsigned)iy < (unsigned)g.h && (unsigned)ix < (unsigned)g.w && row < p.rows;
    ra[slot] = __builtin_amdgcn_raw_buffer_load_b128(
        dy_rsrc, a_ok ? (a_row + (unsigned)__mul24(at, g.fp) + a_col) * (unsigned)sizeof(T) : kOutside, 0, 0);
    rb[slot] = __builtin_amdgcn_raw_buffer_load_b128(
        x_rsrc, b_ok ? (b_row + (unsigned)__mul24(ix, g.cp) + b_col) * (unsigned)sizeof(T) : kOutside, 0, 0);
    at += p.adv_at;
    const bool next = at >= p.period;
    at -= next ? p.period : 0;
    row += p.adv_row + (next ? 1 : 0);
    a_row += a_step + (next ? a_line : 0);
    iy += p.adv_oy * g.stride_h + (next ? g.stride_h : 0);
    b_row += b_step + (next ? b_next : 0);
    const bool image = iy >= iy_end;
    iy -= image ? g.oh * g.stride_h : 0;
    b_row += image ? b_image : 0;
  };
  auto store = [&](int slot, char* stage) {
    *reinterpret_cast<u32x4*>(stage + Tile::LdsOffset(tid, 0))           = ra[slot];
    *reinterpret_cast<u32x4*>(stage + A_BYTES + Tile::LdsOffset(tid, 0)) = rb[slot];
  };

  flex::f32x4 acc[TM][kTaps][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int q = 0; q < kTaps; ++q)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][q][j] = flex::f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int group = ((lane >> 4) & 1) * 2 + (lane >> 5);  // the eight k of this lane, as Mma::Fragment takes them
  auto multiply = [&](const char* stage) {
    vec8 a[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) a[i] = M::template Fragment<false, BM>(stage, wm * (BM / 2) + i * 16, kg, lane);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      flex::s16x4 part[3];
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const int k = kg * 32 + 8 * group + 4 * r + ((lane & 15) >> 2), n = wn * 32 + j * 16 + 4 * (lane & 3);
        const char* at = stage + A_BYTES + Tile::RowOffset(k, n >> 3) + (n & 7) * 2;
        part[r] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((flex::s16x4 __attribute__((address_space(3)))*)at);
      }
      const flex::s16x8 low  = __builtin_shufflevector(part[0], part[1], 0, 1, 2, 3, 4, 5, 6, 7);
      const flex::s16x8 high = __builtin_shufflevector(part[2], part[2], 0, 1, 2, 3, 0, 1, 2, 3);
      const vec8 b[kTaps]    = {__builtin_bit_cast(vec8, low), __builtin_bit_cast(vec8, __builtin_shufflevector(low, high, 1, 2, 3, 4, 5, 6, 7, 8)),
                                __builtin_bit_cast(vec8, __builtin_shufflevector(low, high, 2, 3, 4, 5, 6, 7, 8, 9))};
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < kTaps; ++q) acc[i][q][j] = flex::Half16<T>::mfma(a[i], b[q], acc[i][q][j]);
    }
  };

  // the rows behind a step's tile of x, which meet dy's zeros: zero as well, once
  if (tid < 2 * (B_ROWS - 64) * 8) {
    const int i = tid & 31;
    *reinterpret_cast<u32x4*>(lds + (tid >> 5) * STAGE + A_BYTES + Tile::RowOffset(64 + (i >> 3), i & 7)) = u32x4{0, 0, 0, 0};
  }
#pragma unroll
  for (int u = 0; u < PF; ++u) load(u);
  store(0, lds);
  __syncthreads();
  // a ring of PF steps in registers (flex::KLoop's); steps behind the last one are requested too: they are outside, or
  // pixels of the next split, and are not multiplied
  for (int s = s0; s < s1; s += PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      if (s + u >= s1) break;
      load(u);
      multiply(lds + (u & 1) * STAGE);
      store((u + 1) % PF, lds + ((u + 1) & 1) * STAGE);
      __syncthreads();
    }
  }

  // the tile through LDS, the two halves of K added there
  float* st    = reinterpret_cast<float*>(lds);
  float* plane = g.planes + (int64_t)split * g.f * g.taps * g.cp;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if (kg == half) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < kTaps; ++q)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              float* to = st + (wm * 32 + i * 16 + 4 * (lane >> 4) + r) * SLD + q * BN + wn * 32 + j * 16 + (lane & 15);
              *to       = half == 0 ? acc[i][q][j][r] : *to + acc[i][q][j][r];
            }
    }
    __syncthreads();
  }
#pragma unroll 1
  for (int i = tid; i < BM * COLS / 8; i += 512) {
    const int f = i / (COLS / 8), col = i % (COLS / 8), q = col / (BN / 8), c = c0 + col % (BN / 8) * 8;
    if (m0 + f >= g.f || kx0 + q >= g.kw || c >= g.cp) continue;
    const float* from = &st[f * SLD + col * 8];
    float* to         = plane + ((int64_t)(m0 + f) * g.taps + ky * g.kw + kx0 + q) * g.cp + c;
    *reinterpret_cast<flex::f32x4*>(to)     = *reinterpret_cast<const flex::f32x4*>(from);
    *reinterpret_cast<flex::f32x4*>(to + 4) = *reinterpret_cast<const flex::f32x4*>(from + 4);
  }
}

// One element of the filter gradient by all threads of a block, pixels outside the image left out instead of multiplied by
// zero; every thread gets the sum.
template <typename T>
__device__ float FilterElement(const FilterGradParams& p, int filter, int tap, int ch, float* shared) {
  const T *x = static_cast<const T*>(p.x), *dy = static_cast<const T*>(p.dy);
  const int ty = tap / p.kw * p.dil_h - p.pad_h, tx = tap % p.kw * p.dil_w - p.pad_w;
  float sum = 0.0f;
  for (int first = 0; first < p.pixels; first += 4096) {
    for (int q = first + threadIdx.x; q < min(first + 4096, p.pixels); q += 256) {
      const int n = q / (p.oh * p.ow), rest = q - n * (p.oh * p.ow), oy = rest / p.ow, ox = rest - oy * p.ow;
      const int iy = oy * p.stride_h + ty, ix = ox * p.stride_w + tx;
      if ((unsigned)iy < (unsigned)p.h && (unsigned)ix < (unsigned)p.w)
        sum = __builtin_fmaf((float)dy[(int64_t)q * p.fp + filter], (float)x[((int64_t)n * p.h * p.w + iy * p.w + ix) * p.cp + ch], sum);
    }
    if (__syncthreads_or(sum != sum)) break;  // NaN, whatever else there is
  }
  shared[threadIdx.x] = sum;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) shared[threadIdx.x] += shared[threadIdx.x + k];
    __syncthreads();
  }
  sum = shared[0];
  __syncthreads();
  return sum;
}

// Adds the planes and writes dw: a block takes 64 groups of four columns, its four rows of threads every fourth plane.
// Where a tap lies outside the image the product has multiplied dy by zero, which an infinite or NaN dy makes NaN although
// the sum has no such term: NaNs of such taps are computed again, without those terms.
template <typename T>
__global__ void __launch_bounds__(256)
filter_reduce_kernel(FilterGradParams p, T* __restrict__ dw, int c, int splits, int nhwc, float alpha, float beta) {
  __shared__ __attribute__((aligned(16))) float part[3][64][4];
  __shared__ float shared[256];
  __shared__ int again[64], any;
  const int lane = threadIdx.x & 63, row = threadIdx.x >> 6;
  const int plane = p.f * p.taps * p.cp, at = (blockIdx.x * 64 + lane) * 4;  // below 2^30
  flex::f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
  if (at < plane) {
#pragma unroll 4
    for (int s = row; s < splits; s += 4) v += *reinterpret_cast<const flex::f32x4*>(p.planes + (int64_t)s * plane + at);
  }
  if (row > 0) *reinterpret_cast<flex::f32x4*>(part[row - 1][lane]) = v;
  __syncthreads();
  const int column = at / p.cp, ch = at - column * p.cp, filter = column / p.taps, tap = column - filter * p.taps;
  if (row == 0) {
    int mask = 0;
    if (at < plane) {
#pragma unroll
      for (int r = 0; r < 3; ++r) v += *reinterpret_cast<const flex::f32x4*>(part[r][lane]);
      const int y0 = tap / p.kw * p.dil_h - p.pad_h, x0 = tap % p.kw * p.dil_w - p.pad_w;
      if (p.spill || y0 < 0 || x0 < 0 || y0 + (p.oh - 1) * p.stride_h >= p.h || x0 + (p.ow - 1) * p.stride_w >= p.w) {
#pragma unroll
        for (int e = 0; e < 4; ++e) mask |= v[e] != v[e] && ch + e < c ? 1 << e : 0;
      }
    }
    again[lane] = mask;
    const bool some = __any(mask != 0);
    if (lane == 0) any = some;
  }
  __syncthreads();
  if (any) {
    for (int l = 0; l < 64; ++l) {
      const int other = (blockIdx.x * 64 + l) * 4, col = other / p.cp;
      for (int e = 0; e < 4; ++e) {
        if (!(again[l] >> e & 1)) continue;
        const float sum = FilterElement<T>(p, col / p.taps, col % p.taps, other % p.cp + e, shared);
        if (row == 0 && lane == l) v[e] = sum;
      }
    }
  }
  if (row > 0 || at >= plane) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (ch + e >= c) break;
    const int64_t o = nhwc ? ((int64_t)filter * p.taps + tap) * c + ch + e : ((int64_t)filter * c + ch + e) * p.taps + tap;
    float g = alpha * v[e];
    if (beta != 0.0f) g += beta * (float)dw[o];
    dw[o] = (T)g;
  }
}

// ---- host ----------------------------------------------------------------------------------------------------------
int ChunkElems(const cinn_type_t& t) { return 16 / (t.bits / CHAR_BIT); }
int RoundUp(int v, int to) { return (v + to - 1) / to * to; }
bool Aligned(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

bool TypeSupported(const cinn_type_t& t) {
  return (t.code == cinn_type_float && (t.bits == 16 || t.bits == 32)) || (t.code == cinn_type_bfloat && t.bits == 16);
}

template <typename T>
void Pack(const void* in, void* out, bool nhwc, int n, int c, int plane, int cp, hipStream_t stream) {
  const dim3 grid((plane + 63) / 64, (cp + 63) / 64, n);
  if (nhwc) {
    hipLaunchKernelGGL((pack_kernel<T, false>), grid, dim3(256), 0, stream, static_cast<const T*>(in), static_cast<T*>(out), c, plane, cp);
  } else {
    hipLaunchKernelGGL((pack_kernel<T, true>), grid, dim3(256), 0, stream, static_cast<const T*>(in), static_cast<T*>(out), c, plane, cp);
  }
}

// Both are false, with nothing launched, while the stream is captured and its scratch is too small for the copies and
// planes, or the page of zeros does not exist yet: the gather kernels, which need none, take such a call.
template <typename T>
bool Data(const ConvBackwardArgs& a, hipStream_t stream) {
  constexpr int E = 16 / (int)sizeof(T);
  const int fp        = RoundUp(a.f, E);
  const bool pack_dy  = !a.nhwc || fp != a.f || !Aligned(a.dy);
  const bool unpack   = !a.nhwc && (a.c > 1 && a.h * a.w_in > 1);
  const bool forward  = a.stride_h == 1 && a.stride_w == 1 && (a.kh - 1) * a.dil_h >= a.pad_h && (a.kw - 1) * a.dil_w >= a.pad_w;
  const int classes   = forward ? 1 : a.stride_h * a.stride_w;
  const int slots_w   = forward ? 1 : std::min(a.kw, a.stride_w);
  const int slots     = forward ? 1 : std::min(a.kh, a.stride_h) * slots_w;  // classes that have taps
  const int64_t slot  = (int64_t)RoundUp(a.c * ((a.kh + a.stride_h - 1) / a.stride_h) * ((a.kw + a.stride_w - 1) / a.stride_w) * fp, 128);
  auto bytes = [](int64_t elems) { return ((size_t)elems * sizeof(T) + 255) & ~(size_t)255; };
  const size_t dy_bytes = pack_dy ? bytes((int64_t)a.n * a.oh * a.ow * fp) : 0;
  const size_t wt_bytes = bytes(slots * slot);
  const size_t dx_bytes = unpack ? bytes((int64_t)a.n * a.h * a.w_in * a.c) : 0;
  if (!HasZeroPage(stream) || dy_bytes + wt_bytes + dx_bytes > ScratchLimit(ScratchKind::kTranspose, stream)) return false;
  char* scratch = static_cast<char*>(Scratch(ScratchKind::kTranspose, dy_bytes + wt_bytes + dx_bytes, stream));
  const void* dy = a.dy;
  if (pack_dy) {
    Pack<T>(a.dy, scratch, a.nhwc, a.n, a.f, a.oh * a.ow, fp, stream);
    dy = scratch;
  }
  void* wt = scratch + dy_bytes;
  void* dx = unpack ? scratch + dy_bytes + wt_bytes : a.out;
  FilterParams fpar{a.f, a.c, a.kh, a.kw, fp, a.nhwc ? 1 : 0, forward ? 1 : a.stride_h, forward ? 1 : a.stride_w, slots_w, forward ? 1 : 0, slot};
  hipLaunchKernelGGL(filter_kernel<T>, dim3((unsigned)((slot + 255) / 256), slots), dim3(256), 0, stream,
                     static_cast<const T*>(a.w), static_cast<T*>(wt), fpar);
  // what the gradient is added to goes into the copy first: the sum is rounded once, in the product's epilogue
  if (unpack && a.beta != 0.0f) Pack<T>(a.out, dx, false, a.n, a.c, a.h * a.w_in, a.c, stream);
  if (forward) {
    ConvNhwcArgs c;
    c.x = dy, c.w = wt, c.y = dx;
    c.scale = c.shift = nullptr;
    c.residual       = a.beta != 0.0f ? dx : nullptr;
    c.alpha          = a.alpha;
    c.residual_scale = a.beta;
    c.relu = c.nchw_input = false;
    c.n = a.n, c.h = a.oh, c.w_in = a.ow, c.c = fp;
    c.oc = a.c, c.kh = a.kh, c.kw = a.kw, c.oh = a.h, c.ow = a.w_in;
    c.pad_h = (a.kh - 1) * a.dil_h - a.pad_h, c.pad_w = (a.kw - 1) * a.dil_w - a.pad_w;
    c.stride_h = c.stride_w = 1;
    c.dil_h = a.dil_h, c.dil_w = a.dil_w;
    c.type = a.type;
    c.whole_without_scratch = true;
    RunConvNhwc(c, stream);
  } else {
    DataParams p{dy, wt, dx, ZeroPage(), a.n, a.h, a.w_in, a.c, a.oh, a.ow, fp, a.kh, a.kw, a.stride_h, a.stride_w, a.pad_h, a.pad_w,
                 slots_w, slot, a.alpha, a.beta};
    const int rows = a.n * ((a.h + a.stride_h - 1) / a.stride_h) * ((a.w_in + a.stride_w - 1) / a.stride_w);
    auto tiles = [&](int t) { return (unsigned)(((rows + t - 1) / t) * ((a.c + t - 1) / t)); };
    bool large = false;
    if constexpr (sizeof(T) == 2) {
      // Two blocks of 128x128 on every CU; fewer are better off as four times as many small ones.  us on 64x64 | 128x128
      // tiles, fp16, by the number of the latter (all classes): 84 (96 -> 200 3x3 on 35x35) 13.5 | 21.0, 208 (512 -> 512 on
      // 14x14) 42.2 | 51.9, 392 (256 -> 256 on 28x28) 29.7 | 30.3, 784 (128 -> 128 on 56x56) 30.0 | 29.5, 1568 (256 -> 512 1x1
      // on 56x56, three classes of four without a tap) 37.5 | 32.7, 3136 (128 -> 64 on 112x112) 71.7 | 58.1.  64 channels
      // fill half of such a tile: 784 (64 -> 128 on 56x56) 19.4 | 27.1.
      if (tiles(128) * classes >= 512) {
        hipLaunchKernelGGL((conv_data_kernel<T, 128, 128>), dim3(tiles(128), classes), dim3(256), 0, stream, p);
        large = true;
      }
    }
    if (!large) hipLaunchKernelGGL((conv_data_kernel<T, 64, 64>), dim3(tiles(64), classes), dim3(256), 0, stream, p);
  }
  if (unpack) {
    const int plane = a.h * a.w_in;
    hipLaunchKernelGGL((unpack_kernel<T>), dim3((plane + 63) / 64, (a.c + 63) / 64, a.n), dim3(256), 0, stream,
                       static_cast<const T*>(dx), static_cast<T*>(a.out), a.c, plane);
  }
  CINN_HIP_CALL(hipGetLastError());
  return true;
}

// Estimates of a filter gradient's two kernels in 16 bits, us: the start, the K steps of a block, the planes.  Fitted to 420 layers,
// channels last, 3x3 to 7x7, 8 to 512 channels and filters (error 4 to 7% of the time on average).  A step of conv_filter_kernel's takes longer
// the more blocks a CU has (at most three of 64 rows, two of 128), one of conv_filter_taps_kernel's, of one block per CU, as
// long as it takes.
double FilterMicroseconds(int rows, int64_t blocks, int steps, double plane_mb) {
  const int full = rows == 64 ? 3 : 2, per_cu = (int)std::min<int64_t>((blocks + 255) / 256, full);
  const double step64[3] = {0.66, 1.0, 1.54}, step128[2] = {0.88, 1.2};
  const double rounds = (double)((blocks + 256 * full - 1) / (256 * full));
  return (rows == 64 ? 6.3 + 0.64 * plane_mb : 7.1 + 0.5 * plane_mb) + rounds * steps * (rows == 64 ? step64 : step128)[per_cu - 1];
}
double TapsMicroseconds(int64_t blocks, int steps, double plane_mb) {
  return 7.2 + 0.81 * plane_mb + (double)((blocks + 255) / 256) * steps * 0.51;
}

// Whether a filter gradient goes to conv_filter_taps_kernel, and its launch: where it needs a fifth less out of L2 than
// conv_filter_kernel's tiles (`p`, `bm` rows each, `splits` of K; `tile_bytes`) and is estimated to be faster.
// Measured, us with the reduction of the planes, conv_filter_kernel | here, fp16, 3x3 unless noted: 64 -> 64 on 56x56, batch 32, 33.3 | 23.6,
// 296 -> 24 on 11x88, batch 32, 30.0 | 24.0, 96 -> 40 on 56x60, batch 25, 36.5 | 30.0, 184 -> 56 7x7 on 53x21, batch 7, 35.5 | 31.7; not taken: short
// ones, 80 -> 8 on 24x31, 8.6 | 10.4, and those whose tiles leave a part of the CUs without a block, 504 -> 136 on 42x18, batch 20, 61.5 |
// 80.0 (144 blocks), 424 -> 48 5x5 on 58x37, batch 15, 103 | 149 (140), 392 -> 8 7x7 on 74x96, batch 6, 214 | 353 (147).  Of 167 layers that read a
// fifth less, 60 are taken: 10% faster on average, the worst 6% slower.
template <typename T>
bool PlanTaps(const ConvBackwardArgs& a, const FilterGradParams& p, int bm, int old_splits, int64_t plane, int64_t tile_bytes, TapsParams* t) {
  if (sizeof(T) != 2 || a.stride_w != 1 || a.dil_w != 1 || a.kw < kTaps) return false;
  // positions in a row are multiplied as signed 24-bit numbers (__mul24); channels are below 2^20
  if (std::max(a.ow, a.w_in) > (1 << 23)) return false;
  // Only filters of which at most one tap stays inside the image for all pixels: an infinite or NaN x meets zeros of dy here, so
  // NaNs of every tap are computed again, a block per element, where the other kernel leaves those of such taps as they are.  A step
  // whose dy overflowed has nothing else: 64 -> 64 3x3 on 56x56, batch 32, channels last, without padding, us, that kernel | here, finite dy 32.8 | 23.8,
  // all NaN 32.6 | 1845 (padded 1802 | 1837).
  auto inside = [](int taps, int dil, int stride, int pad, int out, int size) {
    int count = 0;
    for (int k = 0; k < taps; ++k) count += k * dil >= pad && k * dil - pad + (out - 1) * stride < size ? 1 : 0;
    return (int64_t)count;
  };
  if (inside(a.kh, a.dil_h, a.stride_h, a.pad_h, a.oh, a.h) * inside(a.kw, a.dil_w, a.stride_w, a.pad_w, a.ow, a.w_in) > 1) return false;
  t->g         = p;
  t->g.tiles_m = (a.f + 63) / 64;
  t->tiles_c   = (p.cp + 63) / 64;
  t->groups    = (a.kw + kTaps - 1) / kTaps;
  t->period    = a.ow + kTaps - 1;
  t->rows      = a.n * a.oh;
  t->g.steps   = (int)(((int64_t)t->rows * t->period + kFresh - 1) / kFresh);
  const int64_t tiles = (int64_t)t->g.tiles_m * t->tiles_c * t->groups * a.kh;
  if (tiles * t->g.steps * (64 + 64) * 128 * 5 > tile_bytes * 4) return false;
  t->tiles  = (int)tiles;
  t->adv_at = kFresh % t->period, t->adv_row = kFresh / t->period;
  t->adv_oy = t->adv_row % a.oh, t->adv_n = t->adv_row / a.oh;
  // One block per CU, at least four K steps each, at most 64 MiB of planes.  Two blocks per CU write and read twice the
  // planes: the steps above 127.0, 84.4, 88.8, 65.7, 103.2 and 98.4 us.  (128 filters per block: 128 -> 128 91.9, 256 -> 256 89.1.)
  int splits = std::max(1, std::min(256 / t->tiles, t->g.steps / 4));
  splits     = (int)std::min<int64_t>(splits, std::max<int64_t>(1, ((int64_t)16 << 20) / plane));
  t->lanes_log2 = splits >= 8 ? 3 : splits >= 4 ? 2 : splits >= 2 ? 1 : 0;
  t->splits     = splits >> t->lanes_log2 << t->lanes_log2;
  t->g.steps_per_split = (t->g.steps + t->splits - 1) / t->splits;
  const double mb = (double)plane * sizeof(float) * 1e-6;
  return TapsMicroseconds(tiles * t->splits, t->g.steps_per_split, t->splits * mb) <
         FilterMicroseconds(bm, (int64_t)p.tiles_m * p.tiles_n * old_splits, p.steps_per_split, old_splits * mb);
}

template <typename T>
bool Filter(const ConvBackwardArgs& a, hipStream_t stream) {
  constexpr int E = 16 / (int)sizeof(T), KS = 8 * E;
  const int fp = RoundUp(a.f, E), cp = RoundUp(a.c, E);
  const bool pack_dy = !a.nhwc || fp != a.f || !Aligned(a.dy);
  const bool pack_x  = !a.nhwc || cp != a.c || !Aligned(a.x);
  auto bytes = [](int64_t elems) { return ((size_t)elems * sizeof(T) + 255) & ~(size_t)255; };
  const size_t dy_bytes = pack_dy ? bytes((int64_t)a.n * a.oh * a.ow * fp) : 0;
  const size_t x_bytes  = pack_x ? bytes((int64_t)a.n * a.h * a.w_in * cp) : 0;
  FilterGradParams p;
  p.f = a.f, p.fp = fp, p.cp = cp, p.h = a.h, p.w = a.w_in, p.oh = a.oh, p.ow = a.ow, p.kw = a.kw, p.taps = a.kh * a.kw;
  p.stride_h = a.stride_h, p.stride_w = a.stride_w, p.pad_h = a.pad_h, p.pad_w = a.pad_w, p.dil_h = a.dil_h, p.dil_w = a.dil_w;
  p.pixels = a.n * a.oh * a.ow;
  p.steps  = (p.pixels + KS - 1) / KS;
  p.adv_n  = KS / (a.oh * a.ow);
  p.adv_oy = KS / a.ow % a.oh;
  p.adv_ox = KS % a.ow;
  const int columns = p.taps * cp;
  const int bm = sizeof(T) == 2 && a.f > 64 ? 128 : 64;
  const int bn = sizeof(T) == 2 && columns > 64 ? 128 : 64;
  p.tiles_m = (a.f + bm - 1) / bm;
  p.tiles_n = (columns + bn - 1) / bn;
  const int tiles = p.tiles_m * p.tiles_n;
  // Blocks for two to three rounds of the chip, at least four K steps each, at most 64 MiB of planes.  us with 256 | 512 |
  // 768 | 1024 blocks, 3x3 at batch 32: fp16, 128 rows: 128 -> 128 on 28x28 29.0 | 30.7 | 38.4 | 41.2, 256 -> 256 on 14x14
  // 27.8 | 27.7 | 32.4 | 32.3, 512 -> 512 on 7x7 43.0 | 33.2 | 38.3 | 38.3; 64 rows: 64 -> 64 on 56x56 31.8 | 30.3 | 34.2 |
  // 36.9; fp32: 64 -> 64 on 56x56 96 | 81 | 79 | 80, 256 -> 256 on 14x14 154 | 92 | 83 | 79.
  const int64_t plane = (int64_t)a.f * columns;
  int splits = std::max(1, (bm == 128 ? 512 : 768) / tiles);
  splits     = std::min(splits, std::max(1, p.steps / 4));
  splits     = (int)std::min<int64_t>(splits, std::max<int64_t>(1, ((int64_t)16 << 20) / plane));
  p.steps_per_split = (p.steps + splits - 1) / splits;
  splits            = (p.steps + p.steps_per_split - 1) / p.steps_per_split;
  TapsParams t;
  const bool taps = PlanTaps<T>(a, p, bm, splits, plane, (int64_t)tiles * p.steps * (bm + bn) * 128, &t);
  if (taps) splits = t.splits;
  p.spill = taps ? 1 : 0;
  const size_t plane_bytes = (size_t)splits * plane * sizeof(float);
  if (!HasZeroPage(stream) || dy_bytes + x_bytes > ScratchLimit(ScratchKind::kTranspose, stream) ||
      plane_bytes > ScratchLimit(ScratchKind::kSplitK, stream))
    return false;
  char* scratch = dy_bytes + x_bytes ? static_cast<char*>(Scratch(ScratchKind::kTranspose, dy_bytes + x_bytes, stream)) : nullptr;
  p.planes = static_cast<float*>(Scratch(ScratchKind::kSplitK, plane_bytes, stream));
  p.dy = a.dy, p.x = a.x, p.zeros = ZeroPage();
  if (pack_dy) {
    Pack<T>(a.dy, scratch, a.nhwc, a.n, a.f, a.oh * a.ow, fp, stream);
    p.dy = scratch;
  }
  if (pack_x) {
    Pack<T>(a.x, scratch + dy_bytes, a.nhwc, a.n, a.c, a.h * a.w_in, cp, stream);
    p.x = scratch + dy_bytes;
  }
  const dim3 grid(tiles, splits);
  bool done = false;
  if constexpr (sizeof(T) == 2) {
    done = true;
    if (taps) {
      t.g.dy = p.dy, t.g.x = p.x, t.g.planes = p.planes;
      hipLaunchKernelGGL((conv_filter_taps_kernel<T>), dim3((unsigned)(t.tiles * t.splits)), dim3(512), 0, stream, t);
    } else if (bm == 128 && bn == 128) {
      hipLaunchKernelGGL((conv_filter_kernel<T, 128, 128>), grid, dim3(256), 0, stream, p);
    } else if (bm == 128) {
      hipLaunchKernelGGL((conv_filter_kernel<T, 128, 64>), grid, dim3(256), 0, stream, p);
    } else if (bn == 128) {
      hipLaunchKernelGGL((conv_filter_kernel<T, 64, 128>), grid, dim3(256), 0, stream, p);
    } else {
      done = false;
    }
  }
  if (!done) hipLaunchKernelGGL((conv_filter_kernel<T, 64, 64>), grid, dim3(256), 0, stream, p);
  hipLaunchKernelGGL((filter_reduce_kernel<T>), dim3((unsigned)((plane / 4 + 63) / 64)), dim3(256), 0, stream, p,
                     static_cast<T*>(a.out), a.c, splits, a.nhwc ? 1 : 0, a.alpha, a.beta);
  CINN_HIP_CALL(hipGetLastError());
  return true;
}

// Everything is addressed with 32-bit element offsets, also with the channels rounded up.  An empty batch or output (there
// is nothing to divide into steps then) and a negative padding (remainder classes are counted from 0) are left to the
// gather kernels.
bool Fits(const ConvBackwardArgs& a) {
  if (std::min({a.n, a.c, a.h, a.w_in, a.f, a.kh, a.kw, a.oh, a.ow}) < 1 || a.pad_h < 0 || a.pad_w < 0) return false;
  const int e = ChunkElems(a.type);
  const int64_t cp = RoundUp(a.c, e), fp = RoundUp(a.f, e), limit = INT_MAX / 2;
  return TypeSupported(a.type) && a.n <= 65535 && a.n * (int64_t)a.h * a.w_in * cp < limit && a.n * (int64_t)a.oh * a.ow * fp < limit &&
         cp * a.kh * a.kw * fp < limit && cp < (1 << 20) && fp < (1 << 20);
}

}  // namespace

bool TryConvBackwardData(const ConvBackwardArgs& a, hipStream_t stream) {
  if (!Fits(a)) return false;
  const bool forward = a.stride_h == 1 && a.stride_w == 1 && (a.kh - 1) * a.dil_h >= a.pad_h && (a.kw - 1) * a.dil_w >= a.pad_w;
  if (!forward && (a.dil_h != 1 || a.dil_w != 1 || a.stride_h * a.stride_w > 1024)) return false;
  if (a.type.code == cinn_type_bfloat) return Data<__bf16>(a, stream);
  if (a.type.bits == 16) return Data<_Float16>(a, stream);
  return Data<float>(a, stream);
}

bool TryConvBackwardFilter(const ConvBackwardArgs& a, hipStream_t stream) {
  if (!Fits(a)) return false;
  if (a.type.code == cinn_type_bfloat) return Filter<__bf16>(a, stream);
  if (a.type.bits == 16) return Filter<_Float16>(a, stream);
  return Filter<float>(a, stream);
}

}  // namespace cinn_hip_kernels
