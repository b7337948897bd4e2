// Backward intrinsics of the vendor-library call sites: cinn_call_cudnn_conv2d_backward_data /
// cinn_call_cudnn_conv2d_backward_filter (cinn/runtime/cuda/cuda_util.cc:722-967), cinn_call_cudnn_pool2d_backward
// (1043-1119) and cinn_call_cudnn_softmax_backward (1169-1217).  Same argument lists and tensor formats
// (0 = NCHW with [F][C][KH][KW] filters, 1 = NHWC with [F][KH][KW][C] filters), results
// out = alpha * gradient + beta * out, fp32 accumulation for fp32 / fp16 / bf16 tensors, fp64 for fp64 tensors.
//
// Convolution gradients without groups in fp32 / fp16 / bf16 run on the matrix cores (conv_backward_mfma.hip).  The
// kernels here are the straightforward gather forms - one thread (or, for the filter gradient, one block) per gradient
// element, summing its contributions in a fixed order: convolutions with groups, fp64, pooling and log-softmax.
//   dx[n,c,iy,ix] = sum over f of the group, ky, kx with iy = oy * stride - pad + ky * dilation (same in x):
//                   dy[n,f,oy,ox] * w[f,c',ky,kx]
//   dw[f,c',ky,kx] = sum over n, oy, ox: x[n,c,oy * stride - pad + ky * dilation, ...] * dy[n,f,oy,ox]
//   max pooling: the gradient of a window goes to its first maximum in (ky, kx) order (x == y decides, as the
//                library compares the forward output with the input); average pooling divides by kh * kw (mode 1)
//                or by the number of window positions inside the input (mode 2)
//   log-softmax (the only algorithm the reference requests): dx = dy - exp(y) * sum(dy) over the softmax axis
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "cinn_hip_runtime.h"
#include "kernels/conv_backward.h"
#include "runtime/hip_check.h"

namespace {

cinn_buffer_t* Arg(void* v_args, int index) {
  auto* args = static_cast<cinn_pod_value_t*>(v_args);
  CINN_RT_CHECK(args[index].type_code_ == CINN_POD_BUFFER_P, "argument %d is not a buffer", index);
  return static_cast<cinn_buffer_t*>(args[index].value_.v_handle);
}

enum class Elem { kF32, kF16, kBF16, kF64 };
Elem ElemOf(const cinn_buffer_t* b) {
  const int bytes = b->type.bits / CHAR_BIT;
  if (b->type.code == cinn_type_float && bytes == 8) return Elem::kF64;
  if (b->type.code == cinn_type_float && bytes == 4) return Elem::kF32;
  if (b->type.code == cinn_type_float && bytes == 2) return Elem::kF16;
  if (b->type.code == cinn_type_bfloat) return Elem::kBF16;
  fprintf(stderr, "backward intrinsic: unsupported data type code %d bits %d\n", b->type.code, b->type.bits);
  abort();
}

// the type sums are kept in
template <typename T>
struct AccOf {
  typedef float type;
};
template <>
struct AccOf<double> {
  typedef double type;
};
__device__ __forceinline__ float Fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double Fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

struct ConvDims {
  int n, c, ih, iw;      // input
  int f, fc, kh, kw;     // filter: f output channels, fc = c / groups input channels each
  int oh, ow;
  int ph, pw, sh, sw, dh, dw, groups;
  int nhwc;
  float alpha, beta;
};

// element offsets in either format
__device__ __forceinline__ int64_t TensorAt(int nhwc, int C, int H, int W, int n, int c, int h, int w) {
  return nhwc ? (((int64_t)n * H + h) * W + w) * C + c : (((int64_t)n * C + c) * H + h) * W + w;
}
__device__ __forceinline__ int64_t FilterAt(int nhwc, int FC, int KH, int KW, int f, int c, int ky, int kx) {
  return nhwc ? (((int64_t)f * KH + ky) * KW + kx) * FC + c : (((int64_t)f * FC + c) * KH + ky) * KW + kx;
}

template <typename T>
__global__ void __launch_bounds__(256)
conv_backward_data_kernel(const T* __restrict__ w, const T* __restrict__ dy, T* __restrict__ dx, ConvDims p) {
  const int64_t total = (int64_t)p.n * p.c * p.ih * p.iw;
  const int64_t idx   = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= total) return;
  // idx enumerates dx in its own memory order, so that consecutive threads write consecutive elements
  int n, c, iy, ix;
  if (p.nhwc) {
    c  = (int)(idx % p.c);
    ix = (int)((idx / p.c) % p.iw);
    iy = (int)((idx / ((int64_t)p.c * p.iw)) % p.ih);
    n  = (int)(idx / ((int64_t)p.c * p.iw * p.ih));
  } else {
    ix = (int)(idx % p.iw);
    iy = (int)((idx / p.iw) % p.ih);
    c  = (int)((idx / ((int64_t)p.iw * p.ih)) % p.c);
    n  = (int)(idx / ((int64_t)p.iw * p.ih * p.c));
  }
  const int g = c / p.fc, cl = c - g * p.fc;
  const int fg = p.f / p.groups;
  typedef typename AccOf<T>::type Acc;
  Acc acc = 0;
  for (int fl = 0; fl < fg; ++fl) {
    const int f = g * fg + fl;
    for (int ky = 0; ky < p.kh; ++ky) {
      const int ty = iy + p.ph - ky * p.dh;
      if (ty < 0 || ty % p.sh != 0) continue;
      const int oy = ty / p.sh;
      if (oy >= p.oh) continue;
      for (int kx = 0; kx < p.kw; ++kx) {
        const int tx = ix + p.pw - kx * p.dw;
        if (tx < 0 || tx % p.sw != 0) continue;
        const int ox = tx / p.sw;
        if (ox >= p.ow) continue;
        acc = Fma((Acc)dy[TensorAt(p.nhwc, p.f, p.oh, p.ow, n, f, oy, ox)],
                  (Acc)w[FilterAt(p.nhwc, p.fc, p.kh, p.kw, f, cl, ky, kx)], acc);
      }
    }
  }
  Acc v = (Acc)p.alpha * acc;
  if (p.beta != 0.0f) v += (Acc)p.beta * (Acc)dx[idx];
  dx[idx] = (T)v;
}

// one block per filter-gradient element: the 256 threads stride over (n, oy, ox), partial sums meet in LDS
template <typename T>
__global__ void __launch_bounds__(256)
conv_backward_filter_kernel(const T* __restrict__ x, const T* __restrict__ dy, T* __restrict__ dw, ConvDims p) {
  typedef typename AccOf<T>::type Acc;
  __shared__ Acc partial[256];
  const int64_t e = blockIdx.x;  // dw in its own memory order
  int f, cl, ky, kx;
  if (p.nhwc) {
    cl = (int)(e % p.fc);
    kx = (int)((e / p.fc) % p.kw);
    ky = (int)((e / ((int64_t)p.fc * p.kw)) % p.kh);
    f  = (int)(e / ((int64_t)p.fc * p.kw * p.kh));
  } else {
    kx = (int)(e % p.kw);
    ky = (int)((e / p.kw) % p.kh);
    cl = (int)((e / ((int64_t)p.kw * p.kh)) % p.fc);
    f  = (int)(e / ((int64_t)p.kw * p.kh * p.fc));
  }
  const int fg = p.f / p.groups;
  const int c  = (f / fg) * p.fc + cl;
  const int64_t positions = (int64_t)p.n * p.oh * p.ow;
  Acc acc = 0;
  for (int64_t q = threadIdx.x; q < positions; q += 256) {
    const int ox = (int)(q % p.ow);
    const int oy = (int)((q / p.ow) % p.oh);
    const int n  = (int)(q / ((int64_t)p.ow * p.oh));
    const int iy = oy * p.sh - p.ph + ky * p.dh, ix = ox * p.sw - p.pw + kx * p.dw;
    if (iy < 0 || iy >= p.ih || ix < 0 || ix >= p.iw) continue;
    acc = Fma((Acc)x[TensorAt(p.nhwc, p.c, p.ih, p.iw, n, c, iy, ix)],
              (Acc)dy[TensorAt(p.nhwc, p.f, p.oh, p.ow, n, f, oy, ox)], acc);
  }
  partial[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) partial[threadIdx.x] += partial[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    Acc v = (Acc)p.alpha * partial[0];
    if (p.beta != 0.0f) v += (Acc)p.beta * (Acc)dw[e];
    dw[e] = (T)v;
  }
}

struct PoolDims {
  int n, c, ih, iw, oh, ow, kh, kw, ph, pw, sh, sw;
  int mode, nhwc;
  float alpha, beta;
};

template <typename T>
__global__ void __launch_bounds__(256)
pool_backward_kernel(const T* __restrict__ x, const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx,
                     PoolDims p) {
  const int64_t total = (int64_t)p.n * p.c * p.ih * p.iw;
  const int64_t idx   = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= total) return;
  int n, c, iy, ix;
  if (p.nhwc) {
    c  = (int)(idx % p.c);
    ix = (int)((idx / p.c) % p.iw);
    iy = (int)((idx / ((int64_t)p.c * p.iw)) % p.ih);
    n  = (int)(idx / ((int64_t)p.c * p.iw * p.ih));
  } else {
    ix = (int)(idx % p.iw);
    iy = (int)((idx / p.iw) % p.ih);
    c  = (int)((idx / ((int64_t)p.iw * p.ih)) % p.c);
    n  = (int)(idx / ((int64_t)p.iw * p.ih * p.c));
  }
  typedef typename AccOf<T>::type Acc;
  const bool is_max = p.mode == 0 || p.mode == 3;
  const Acc mine    = (Acc)x[idx];
  Acc acc = 0;
  // windows (oy, ox) that contain (iy, ix): oy * sh - ph <= iy < oy * sh - ph + kh.  Only those are visited: a loop over
  // all of them took 25.6 us for [8][18][21][200] fp32 and 3x3 windows two apart, this one 21.4.
  const int top = iy + p.ph, left = ix + p.pw;
  const int oy0 = top < p.kh ? 0 : (top - p.kh) / p.sh + 1, oy1 = top < 0 ? -1 : min(p.oh - 1, top / p.sh);
  const int ox0 = left < p.kw ? 0 : (left - p.kw) / p.sw + 1, ox1 = left < 0 ? -1 : min(p.ow - 1, left / p.sw);
  for (int oy = oy0; oy <= oy1; ++oy) {
    const int ys = oy * p.sh - p.ph;
    for (int ox = ox0; ox <= ox1; ++ox) {
      const int xs = ox * p.sw - p.pw;
      const int64_t o = TensorAt(p.nhwc, p.c, p.oh, p.ow, n, c, oy, ox);
      const Acc g     = (Acc)dy[o];
      if (is_max) {
        const Acc m = (Acc)y[o];
        if (mine != m) continue;
        // the first element of the window (rows, then columns) that equals the maximum takes the gradient
        bool first = true;
        for (int ry = 0; ry < p.kh && first; ++ry) {
          const int yy = ys + ry;
          if (yy < 0 || yy >= p.ih) continue;
          for (int rx = 0; rx < p.kw; ++rx) {
            const int xx = xs + rx;
            if (xx < 0 || xx >= p.iw) continue;
            if (yy == iy && xx == ix) { ry = p.kh; break; }
            if ((Acc)x[TensorAt(p.nhwc, p.c, p.ih, p.iw, n, c, yy, xx)] == m) { first = false; break; }
          }
        }
        if (first) acc += g;
      } else {
        Acc factor = (Acc)(p.kh * p.kw);
        if (p.mode == 2) {
          const int y0 = ys > 0 ? ys : 0, x0 = xs > 0 ? xs : 0;
          const int y1 = ys + p.kh < p.ih ? ys + p.kh : p.ih, x1 = xs + p.kw < p.iw ? xs + p.kw : p.iw;
          const int count = (y1 - y0) * (x1 - x0);
          factor          = (Acc)(count > 1 ? count : 1);
        }
        acc += g / factor;
      }
    }
  }
  Acc v = (Acc)p.alpha * acc;
  if (p.beta != 0.0f) v += (Acc)p.beta * (Acc)dx[idx];
  dx[idx] = (T)v;
}

// Max pooling of 3x3 windows two apart, the pooling of image networks: an element lies in at most two by two windows, and
// has to be compared with what precedes it in each.  The loop above reads those one after another and leaves at the first
// match, a chain of dependent loads; here a window's are in flight together (masked ones read the element itself), and
// channels-last tensors go E elements of 16 bytes per thread, which the index arithmetic is bound by otherwise.
// [8][18][21][200] fp32: 21.4 us in the loop, 17.2 with one element per thread, 9.5 here.
template <typename T, int E>
__global__ void __launch_bounds__(256)
max_pool3s2_backward_kernel(const T* __restrict__ x, const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx,
                            PoolDims p) {
  struct Chunk {
    T v[E];
  };
  auto load = [](const T* from) {
    Chunk c;
    __builtin_memcpy(&c, __builtin_assume_aligned(from, sizeof(Chunk)), sizeof(Chunk));
    return c;
  };
  const int64_t idx = ((int64_t)blockIdx.x * 256 + threadIdx.x) * E;
  if (idx >= (int64_t)p.n * p.c * p.ih * p.iw) return;
  const int at = (int)idx;  // the call takes tensors of fewer than 2^31 elements
  int n, c, iy, ix;
  if (p.nhwc) {
    const int pixel = at / p.c, row = pixel / p.iw;
    c = at - pixel * p.c, ix = pixel - row * p.iw, n = row / p.ih, iy = row - n * p.ih;
  } else {
    const int row = at / p.iw, plane = row / p.ih;
    ix = at - row * p.iw, iy = row - plane * p.ih, n = plane / p.c, c = plane - n * p.c;
  }
  // elements between columns and rows of the input and of the output
  const int step_x = p.nhwc ? p.c : 1, row_x = p.iw * step_x, row_y = p.ow * step_x;
  const int first_y = p.nhwc ? n * p.oh * row_y + c : (n * p.c + c) * p.oh * row_y;
  typedef typename AccOf<T>::type Acc;
  const Chunk mine = load(x + at);
  const int top = iy + p.ph, left = ix + p.pw;  // >= 0: paddings are not negative here
  Acc acc[E];
#pragma unroll
  for (int i = 0; i < E; ++i) acc[i] = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    // in ascending order of windows, as the sums of the general kernel are
    const int oy = top / 2 - 1 + w / 2, ox = left / 2 - 1 + w % 2;
    const int ry = top - 2 * oy, rx = left - 2 * ox;  // where the element lies in the window
    if (!(oy >= 0 && oy < p.oh && ox >= 0 && ox < p.ow && ry < 3 && rx < 3)) continue;
    const int o   = first_y + oy * row_y + ox * step_x;
    const Chunk m = load(y + o), g = load(dy + o);
    Chunk seen[8];
    bool before[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int vy = e / 3 - ry, vx = e % 3 - rx;  // from the element to the window's e-th
      before[e]    = (vy < 0 || (vy == 0 && vx < 0)) && iy + vy >= 0 && ix + vx >= 0 && ix + vx < p.iw;
      seen[e]      = load(x + (before[e] ? at + vy * row_x + vx * step_x : at));
    }
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const Acc top_value = (Acc)m.v[i];
      bool takes          = (Acc)mine.v[i] == top_value;
#pragma unroll
      for (int e = 0; e < 8; ++e) takes = takes && !(before[e] && (Acc)seen[e].v[i] == top_value);
      if (takes) acc[i] += (Acc)g.v[i];
    }
  }
  Chunk out;
  if (p.beta != 0.0f) out = load(dx + at);
#pragma unroll
  for (int i = 0; i < E; ++i) {
    Acc v = (Acc)p.alpha * acc[i];
    if (p.beta != 0.0f) v += (Acc)p.beta * (Acc)out.v[i];
    out.v[i] = (T)v;
  }
  __builtin_memcpy(__builtin_assume_aligned(dx + at, sizeof(Chunk)), &out, sizeof(Chunk));
}

template <typename T>
void LaunchPoolBackward(const cinn_buffer_t* x, const cinn_buffer_t* y, const cinn_buffer_t* dy, const cinn_buffer_t* dx,
                        const PoolDims& p, hipStream_t stream) {
  constexpr int E     = 16 / (int)sizeof(T);
  const int64_t total = (int64_t)p.n * p.c * p.ih * p.iw;
  auto grid           = [&](int per_thread) { return dim3((unsigned)((total + 256 * per_thread - 1) / (256 * per_thread))); };
  const T *xp = reinterpret_cast<const T*>(x->memory), *yp = reinterpret_cast<const T*>(y->memory);
  const T* gp = reinterpret_cast<const T*>(dy->memory);
  T* to       = reinterpret_cast<T*>(dx->memory);
  auto aligned     = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; };
  const bool three = (p.mode == 0 || p.mode == 3) && p.kh == 3 && p.kw == 3 && p.sh == 2 && p.sw == 2 && p.ph >= 0 && p.pw >= 0 &&
                     (int64_t)p.n * p.c * p.oh * p.ow < INT_MAX;
  constexpr int F = sizeof(T) < 4 ? 4 / (int)sizeof(T) : 1;
  if (three && p.nhwc && p.c % E == 0 && aligned(xp) && aligned(yp) && aligned(gp) && aligned(to)) {
    // 4 bytes per thread where 16 would not give 256 CUs a block each: a block by itself is bound by the comparisons of one
    // thread, 9.7 us against 6.6 at [2][15][56] pixels of 32 channels in fp16, and as many more threads cost nothing then.  With
    // the line at 1024 blocks larger tensors lose 3% of a whole training step to the index arithmetic.
    if (total / (256 * E) < 256) {
      hipLaunchKernelGGL((max_pool3s2_backward_kernel<T, F>), grid(F), dim3(256), 0, stream, xp, yp, gp, to, p);
    } else {
      hipLaunchKernelGGL((max_pool3s2_backward_kernel<T, E>), grid(E), dim3(256), 0, stream, xp, yp, gp, to, p);
    }
  } else if (three) {
    hipLaunchKernelGGL((max_pool3s2_backward_kernel<T, 1>), grid(1), dim3(256), 0, stream, xp, yp, gp, to, p);
  } else {
    hipLaunchKernelGGL(pool_backward_kernel<T>, grid(1), dim3(256), 0, stream, xp, yp, gp, to, p);
  }
}

// one block per softmax group: `len` elements `inner` apart
template <typename T>
__global__ void __launch_bounds__(256)
log_softmax_backward_kernel(const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx, int len, int inner,
                            float alpha, float beta) {
  __shared__ float partial[256];
  const int64_t group = blockIdx.x;
  const int64_t base  = (group / inner) * (int64_t)len * inner + group % inner;
  float s = 0.0f;
  for (int i = threadIdx.x; i < len; i += 256) s += (float)dy[base + (int64_t)i * inner];
  partial[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) partial[threadIdx.x] += partial[threadIdx.x + k];
    __syncthreads();
  }
  const float sum = partial[0];
  for (int i = threadIdx.x; i < len; i += 256) {
    const int64_t o = base + (int64_t)i * inner;
    float v         = alpha * ((float)dy[o] - __expf((float)y[o]) * sum);
    if (beta != 0.0f) v += beta * (float)dx[o];
    dx[o] = (T)v;
  }
}

ConvDims MakeConvDims(const char* what, int format, float alpha, float beta, int in, int ic, int ih, int iw, int fn, int fc,
                      int fh, int fw, int ph, int pw, int sh, int sw, int dh, int dw, int groups, int on, int oc, int oh,
                      int ow) {
  CINN_RT_CHECK(format == 0 || format == 1, "%s: unknown tensor format %d", what, format);
  CINN_RT_CHECK(groups >= 1 && ic % groups == 0 && fn % groups == 0, "%s: bad group count %d", what, groups);
  CINN_RT_CHECK(fc == ic / groups, "%s: filter has %d input channels, expected %d", what, fc, ic / groups);
  CINN_RT_CHECK(on == in && oc == fn, "%s: output gradient is [%d,%d,..], expected [%d,%d,..]", what, on, oc, in, fn);
  CINN_RT_CHECK(sh > 0 && sw > 0 && dh > 0 && dw > 0, "%s: strides and dilations must be positive", what);
  const int want_oh = (ih - ((fh - 1) * dh + 1) + 2 * ph) / sh + 1;
  const int want_ow = (iw - ((fw - 1) * dw + 1) + 2 * pw) / sw + 1;
  CINN_RT_CHECK(oh == want_oh && ow == want_ow, "%s: output is %dx%d, the shapes give %dx%d", what, oh, ow, want_oh, want_ow);
  CINN_RT_CHECK((int64_t)in * ic * ih * iw < INT_MAX && (int64_t)on * oc * oh * ow < INT_MAX, "%s: tensor too large", what);
  ConvDims p;
  p.n = in, p.c = ic, p.ih = ih, p.iw = iw;
  p.f = fn, p.fc = fc, p.kh = fh, p.kw = fw;
  p.oh = oh, p.ow = ow;
  p.ph = ph, p.pw = pw, p.sh = sh, p.sw = sw, p.dh = dh, p.dw = dw, p.groups = groups;
  p.nhwc  = format == 1;
  p.alpha = alpha, p.beta = beta;
  return p;
}

cinn_hip_kernels::ConvBackwardArgs MatrixArgs(const ConvDims& p, const cinn_buffer_t* out) {
  cinn_hip_kernels::ConvBackwardArgs a;
  a.x = a.w = a.dy = nullptr;
  a.out  = out->memory;
  a.nhwc = p.nhwc != 0;
  a.n = p.n, a.c = p.c, a.h = p.ih, a.w_in = p.iw;
  a.f = p.f, a.kh = p.kh, a.kw = p.kw, a.oh = p.oh, a.ow = p.ow;
  a.pad_h = p.ph, a.pad_w = p.pw, a.stride_h = p.sh, a.stride_w = p.sw, a.dil_h = p.dh, a.dil_w = p.dw;
  a.alpha = p.alpha, a.beta = p.beta;
  a.type = out->type;
  return a;
}

}  // namespace

extern "C" {

void cinn_call_cudnn_conv2d_backward_data(void* v_args, int num_args, int format, float alpha, float beta, int input_n,
                                          int input_c, int input_h, int input_w, int filter_n, int filter_c,
                                          int filter_h, int filter_w, int pad_h, int pad_w, int stride_h, int stride_w,
                                          int dilation_h, int dilation_w, int groups, int output_n, int output_c,
                                          int output_h, int output_w, void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  CINN_RT_CHECK(num_args == 3, "cinn_call_cudnn_conv2d_backward_data takes w, dy and dx, got %d arguments", num_args);
  const ConvDims p = MakeConvDims("conv2d_backward_data", format, alpha, beta, input_n, input_c, input_h, input_w, filter_n,
                                  filter_c, filter_h, filter_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w,
                                  groups, output_n, output_c, output_h, output_w);
  cinn_buffer_t* w  = Arg(v_args, 0);
  cinn_buffer_t* dy = Arg(v_args, 1);
  cinn_buffer_t* dx = Arg(v_args, 2);
  if (p.groups == 1) {
    cinn_hip_kernels::ConvBackwardArgs a = MatrixArgs(p, dx);
    a.w = w->memory, a.dy = dy->memory;
    if (cinn_hip_kernels::TryConvBackwardData(a, static_cast<hipStream_t>(stream))) return;
  }
  const int64_t total = (int64_t)p.n * p.c * p.ih * p.iw;
  dim3 grid((unsigned)((total + 255) / 256));
  auto s = static_cast<hipStream_t>(stream);
  switch (ElemOf(dx)) {
    case Elem::kF64:
      hipLaunchKernelGGL(conv_backward_data_kernel<double>, grid, dim3(256), 0, s, reinterpret_cast<const double*>(w->memory), reinterpret_cast<const double*>(dy->memory), reinterpret_cast<double*>(dx->memory), p);
      break;
    case Elem::kF32:
      hipLaunchKernelGGL(conv_backward_data_kernel<float>, grid, dim3(256), 0, s, reinterpret_cast<const float*>(w->memory),
                         reinterpret_cast<const float*>(dy->memory), reinterpret_cast<float*>(dx->memory), p);
      break;
    case Elem::kF16:
      hipLaunchKernelGGL(conv_backward_data_kernel<_Float16>, grid, dim3(256), 0, s,
                         reinterpret_cast<const _Float16*>(w->memory), reinterpret_cast<const _Float16*>(dy->memory),
                         reinterpret_cast<_Float16*>(dx->memory), p);
      break;
    case Elem::kBF16:
      hipLaunchKernelGGL(conv_backward_data_kernel<__bf16>, grid, dim3(256), 0, s, reinterpret_cast<const __bf16*>(w->memory),
                         reinterpret_cast<const __bf16*>(dy->memory), reinterpret_cast<__bf16*>(dx->memory), p);
      break;
  }
  CINN_HIP_CALL(hipGetLastError());
}

void cinn_call_cudnn_conv2d_backward_filter(void* v_args, int num_args, int format, float alpha, float beta, int input_n,
                                            int input_c, int input_h, int input_w, int filter_n, int filter_c,
                                            int filter_h, int filter_w, int pad_h, int pad_w, int stride_h,
                                            int stride_w, int dilation_h, int dilation_w, int groups, int output_n,
                                            int output_c, int output_h, int output_w, void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  CINN_RT_CHECK(num_args == 3, "cinn_call_cudnn_conv2d_backward_filter takes x, dy and dw, got %d arguments", num_args);
  const ConvDims p = MakeConvDims("conv2d_backward_filter", format, alpha, beta, input_n, input_c, input_h, input_w,
                                  filter_n, filter_c, filter_h, filter_w, pad_h, pad_w, stride_h, stride_w, dilation_h,
                                  dilation_w, groups, output_n, output_c, output_h, output_w);
  cinn_buffer_t* x  = Arg(v_args, 0);
  cinn_buffer_t* dy = Arg(v_args, 1);
  cinn_buffer_t* dw = Arg(v_args, 2);
  const int64_t total = (int64_t)p.f * p.fc * p.kh * p.kw;
  CINN_RT_CHECK(total < INT_MAX, "conv2d_backward_filter: filter too large");
  if (p.groups == 1) {
    cinn_hip_kernels::ConvBackwardArgs a = MatrixArgs(p, dw);
    a.x = x->memory, a.dy = dy->memory;
    if (cinn_hip_kernels::TryConvBackwardFilter(a, static_cast<hipStream_t>(stream))) return;
  }
  dim3 grid((unsigned)total);
  auto s = static_cast<hipStream_t>(stream);
  switch (ElemOf(dw)) {
    case Elem::kF64:
      hipLaunchKernelGGL(conv_backward_filter_kernel<double>, grid, dim3(256), 0, s, reinterpret_cast<const double*>(x->memory), reinterpret_cast<const double*>(dy->memory), reinterpret_cast<double*>(dw->memory), p);
      break;
    case Elem::kF32:
      hipLaunchKernelGGL(conv_backward_filter_kernel<float>, grid, dim3(256), 0, s, reinterpret_cast<const float*>(x->memory),
                         reinterpret_cast<const float*>(dy->memory), reinterpret_cast<float*>(dw->memory), p);
      break;
    case Elem::kF16:
      hipLaunchKernelGGL(conv_backward_filter_kernel<_Float16>, grid, dim3(256), 0, s,
                         reinterpret_cast<const _Float16*>(x->memory), reinterpret_cast<const _Float16*>(dy->memory),
                         reinterpret_cast<_Float16*>(dw->memory), p);
      break;
    case Elem::kBF16:
      hipLaunchKernelGGL(conv_backward_filter_kernel<__bf16>, grid, dim3(256), 0, s, reinterpret_cast<const __bf16*>(x->memory),
                         reinterpret_cast<const __bf16*>(dy->memory), reinterpret_cast<__bf16*>(dw->memory), p);
      break;
  }
  CINN_HIP_CALL(hipGetLastError());
}

void cinn_call_cudnn_pool2d_backward(void* v_args, int num_args, int mode, int format, float alpha, float beta,
                                     int input_n, int input_c, int input_h, int input_w, int kernel_h, int kernel_w,
                                     int pad_h, int pad_w, int stride_h, int stride_w, int output_n, int output_c,
                                     int output_h, int output_w, void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  CINN_RT_CHECK(num_args == 4, "cinn_call_cudnn_pool2d_backward takes x, y, dy and dx, got %d arguments", num_args);
  CINN_RT_CHECK(format == 0 || format == 1, "pool2d_backward: unknown tensor format %d", format);
  CINN_RT_CHECK(mode >= 0 && mode <= 3, "pool2d_backward: unknown pooling mode %d", mode);
  CINN_RT_CHECK(output_n == input_n && output_c == input_c, "pool2d_backward: batch / channel mismatch");
  CINN_RT_CHECK(kernel_h > 0 && kernel_w > 0 && stride_h > 0 && stride_w > 0 && output_h > 0 && output_w > 0,
                "pool2d_backward: bad window");
  CINN_RT_CHECK((int64_t)input_n * input_c * input_h * input_w < INT_MAX, "pool2d_backward: tensor too large");
  PoolDims p;
  p.n = input_n, p.c = input_c, p.ih = input_h, p.iw = input_w, p.oh = output_h, p.ow = output_w;
  p.kh = kernel_h, p.kw = kernel_w, p.ph = pad_h, p.pw = pad_w, p.sh = stride_h, p.sw = stride_w;
  p.mode = mode, p.nhwc = format == 1;
  p.alpha = alpha, p.beta = beta;
  cinn_buffer_t* x  = Arg(v_args, 0);
  cinn_buffer_t* y  = Arg(v_args, 1);
  cinn_buffer_t* dy = Arg(v_args, 2);
  cinn_buffer_t* dx = Arg(v_args, 3);
  auto s = static_cast<hipStream_t>(stream);
  switch (ElemOf(dx)) {
    case Elem::kF64: LaunchPoolBackward<double>(x, y, dy, dx, p, s); break;
    case Elem::kF32: LaunchPoolBackward<float>(x, y, dy, dx, p, s); break;
    case Elem::kF16: LaunchPoolBackward<_Float16>(x, y, dy, dx, p, s); break;
    case Elem::kBF16: LaunchPoolBackward<__bf16>(x, y, dy, dx, p, s); break;
  }
  CINN_HIP_CALL(hipGetLastError());
}

void cinn_call_cudnn_softmax_backward(void* v_args, int num_args, int mode, int format, float alpha, float beta,
                                      int input_n, int input_c, int input_h, int input_w, int output_n, int output_c,
                                      int output_h, int output_w, void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  CINN_RT_CHECK(num_args == 3, "cinn_call_cudnn_softmax_backward takes y, dy and dx, got %d arguments", num_args);
  CINN_RT_CHECK(format == 0, "softmax_backward: only NCHW (format 0) is implemented, got format %d", format);
  CINN_RT_CHECK(mode == 0 || mode == 1, "softmax_backward: unknown mode %d", mode);
  CINN_RT_CHECK(input_n == output_n && input_c == output_c && input_h == output_h && input_w == output_w,
                "softmax_backward: input and output shapes differ");
  cinn_buffer_t* y  = Arg(v_args, 0);
  cinn_buffer_t* dy = Arg(v_args, 1);
  cinn_buffer_t* dx = Arg(v_args, 2);
  const int len   = mode == 1 ? input_c : input_c * input_h * input_w;
  const int inner = mode == 1 ? input_h * input_w : 1;
  const int64_t groups = (int64_t)input_n * inner;
  CINN_RT_CHECK(groups > 0 && groups < INT_MAX && len > 0, "softmax_backward: bad extents");
  dim3 grid((unsigned)groups);
  auto s = static_cast<hipStream_t>(stream);
  switch (ElemOf(dx)) {
    case Elem::kF64: CINN_RT_CHECK(false, "softmax_backward: fp64 tensors are not implemented"); break;
    case Elem::kF32:
      hipLaunchKernelGGL(log_softmax_backward_kernel<float>, grid, dim3(256), 0, s, reinterpret_cast<const float*>(y->memory),
                         reinterpret_cast<const float*>(dy->memory), reinterpret_cast<float*>(dx->memory), len, inner, alpha, beta);
      break;
    case Elem::kF16:
      hipLaunchKernelGGL(log_softmax_backward_kernel<_Float16>, grid, dim3(256), 0, s,
                         reinterpret_cast<const _Float16*>(y->memory), reinterpret_cast<const _Float16*>(dy->memory),
                         reinterpret_cast<_Float16*>(dx->memory), len, inner, alpha, beta);
      break;
    case Elem::kBF16:
      hipLaunchKernelGGL(log_softmax_backward_kernel<__bf16>, grid, dim3(256), 0, s, reinterpret_cast<const __bf16*>(y->memory),
                         reinterpret_cast<const __bf16*>(dy->memory), reinterpret_cast<__bf16*>(dx->memory), len, inner, alpha, beta);
      break;
  }
  CINN_HIP_CALL(hipGetLastError());
}

}  // extern "C"
