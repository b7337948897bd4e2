// Sums over the pixels of channels-last tensors for gfx950: what a training batch norm needs before it can normalise
// (cinn_call_hip_channel_statistics) and what its gradient needs before it can be formed
// (cinn_call_hip_channel_gradient_sums).
//
// As generated code each sum was a chain of its own - an element-wise kernel that wrote the squares or products to
// memory in fp32, a reduction over runs of pixels, a reduction of those - and the gradient's mask one more pass.  Both
// sums need the same elements, so one pass reads every tensor once and writes nothing of its size: bound by that read.
// A thread owns 16 bytes of channels and walks pixels, four loads in flight; the rows of a block meet in LDS, the
// blocks in a second launch of a few microseconds (the last block to arrive could add them instead, with a counter that it
// sets back; that form has not been measured).
//
// What the sums are for is applied in a second pass (channel_apply_kernel): generated code formed square roots, divisions
// and six per-channel loads for every element and wrote the result through a transpose.
//
// Measured, us, generated -> here: [32][56][56][64] fp16 statistics 36 -> 7.6 (12.8 MB at 3 TB/s and the second launch),
// normalisation with relu 60 (with a transpose, which is now a kernel of 8.2) -> 8.2; gradient with a relu's mask: sums
// 23 -> 11.6, gradient 28 -> 12.5 (51 MB at 4.1 TB/s).  [8][18][21][200] fp32: 9.1, 4.2, 8.7 and 4.6, of which a launch
// is more than half.
//
// All arithmetic is fp32, and every sum is one of short chains: a thread adds its few pixels, then rows and planes are added
// in four chains each, what is left pairwise.  Relative error against float64, generated reductions | one chain each | here:
// mean of [32][56][56][64] fp32 4.1e-8 | 7.3e-8 | 4.0e-8, sum of dy 1.6e-7 | 1.8e-7 | 1.1e-7.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>

#include "cinn_hip_runtime.h"
#include "kernels/flex_tile.h"
#include "runtime/hip_check.h"
#include "runtime/scratch.h"

namespace {

using cinn_hip_kernels::Scratch;
using cinn_hip_kernels::ScratchKind;
using cinn_hip_kernels::ScratchLimit;
using cinn_hip_kernels::flex::LoadAny;

struct SumsParams {
  const void *a, *x, *out;  // a: x itself, or dy
  const float* mean;
  float* planes;  // [split][2][channels], or null: the sums go to first and second
  float *first, *second;
  int64_t pixels;
  int channels, chunk_lanes, pixels_per_split, splits;
};

// mean and E(x^2) - mean^2, each step rounded as the operators round it, of the sums of x and x x
__device__ __forceinline__ void Statistics(float count, float* s, float* t) {
  *s = *s / count;
  *t = __fsub_rn(*t / count, __fmul_rn(*s, *s));
}

// E elements of channels from p: a chunk, or (E = 1) one element
template <typename T, int E>
__device__ __forceinline__ void LoadChannels(const T* p, float (&v)[E]) {
  if constexpr (E == 1) {
    v[0] = (float)*p;
  } else {
    typedef T chunk_t __attribute__((ext_vector_type(E)));
    chunk_t c;
    if constexpr (sizeof(chunk_t) == 16) {
      c = __builtin_bit_cast(chunk_t, LoadAny<T>(reinterpret_cast<const char*>(p)));
    } else {
      __builtin_memcpy(&c, __builtin_assume_aligned(p, sizeof(chunk_t)), sizeof(chunk_t));
    }
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = (float)c[e];
  }
}

// GRAD: sums of dy and dy (x - mean), with dy zero where MASKED and out is not positive; else of x and x x.
// A block takes one split, or (DIRECT) all of them, one after the other, and writes the sums' last form itself.  (As a loop
// that both forms run, the conv_train step of [32][56][56][64] fp16 was 1.3 us of 138 slower.)
template <typename T, int E, bool GRAD, bool MASKED, bool DIRECT>
__global__ void __launch_bounds__(256)
channel_sums_kernel(SumsParams p) {
  __shared__ float meet[256 * 2 * E];
  __shared__ float total[DIRECT ? 2 * E * 64 : 1];
  const int lanes = p.chunk_lanes, rows = 256 / lanes;
  const int tid = threadIdx.x, row = tid / lanes;
  const int ch = (blockIdx.x * lanes + tid % lanes) * E;
  for (int split = blockIdx.y; split < (DIRECT ? p.splits : blockIdx.y + 1); ++split) {
    float s[E], t[E];
#pragma unroll
    for (int e = 0; e < E; ++e) s[e] = t[e] = 0.0f;
    if (ch < p.channels) {
      const int64_t first = (int64_t)split * p.pixels_per_split;
      const int64_t end   = min(first + p.pixels_per_split, p.pixels);
      const T *a = static_cast<const T*>(p.a), *x = static_cast<const T*>(p.x), *o = static_cast<const T*>(p.out);
      float mean[E];
#pragma unroll
      for (int e = 0; e < E; ++e) mean[e] = GRAD ? p.mean[ch + e] : 0.0f;
      auto add = [&](const float (&av)[E], const float (&xv)[E], const float (&ov)[E]) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float d = MASKED ? (ov[e] > 0.0f ? av[e] : 0.0f) : av[e];
          s[e] += d;
          t[e] = __builtin_fmaf(d, GRAD ? xv[e] - mean[e] : d, t[e]);
        }
      };
      constexpr int U = GRAD ? 2 : 4;
      int64_t q       = first + row;
      for (; q + (U - 1) * rows < end; q += U * rows) {
        float av[U][E], xv[U][E], ov[U][E];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t at = (q + u * rows) * p.channels + ch;
          LoadChannels<T, E>(a + at, av[u]);
          if (GRAD) LoadChannels<T, E>(x + at, xv[u]);
          if (MASKED) LoadChannels<T, E>(o + at, ov[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) add(av[u], xv[u], ov[u]);
      }
      for (; q < end; q += rows) {
        float av[E], xv[E], ov[E];
        const int64_t at = q * p.channels + ch;
        LoadChannels<T, E>(a + at, av);
        if (GRAD) LoadChannels<T, E>(x + at, xv);
        if (MASKED) LoadChannels<T, E>(o + at, ov);
        add(av, xv, ov);
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) meet[(2 * e) * 256 + tid] = s[e], meet[(2 * e + 1) * 256 + tid] = t[e];
    __syncthreads();
    // value i = 2 e + (which sum) of lane l: the sum over rows of meet[i][row * lanes + l]
    for (int i = tid; i < 2 * E * lanes; i += 256) {
      const int value = i / lanes, l = i % lanes;
      float q[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // rows: a power of two, at least four
      for (int r = 0; r < rows; r += 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] += meet[value * 256 + (r + u) * lanes + l];
      }
      const float sum = (q[0] + q[1]) + (q[2] + q[3]);
      if constexpr (DIRECT) {
        total[i] = split == 0 ? sum : total[i] + sum;
      } else {
        const int c = (blockIdx.x * lanes + l) * E + value / 2;
        if (c < p.channels) p.planes[((int64_t)split * 2 + (value & 1)) * p.channels + c] = sum;
      }
    }
    if constexpr (DIRECT) __syncthreads();
  }
  if constexpr (!DIRECT) return;
  for (int i = tid; i < E * lanes; i += 256) {
    const int c = (blockIdx.x * lanes + i % lanes) * E + i / lanes;
    float sum = total[2 * (i / lanes) * lanes + i % lanes], other = total[(2 * (i / lanes) + 1) * lanes + i % lanes];
    if (!GRAD) Statistics((float)p.pixels, &sum, &other);
    if (c < p.channels) p.first[c] = sum, p.second[c] = other;
  }
}

// 16 channels per block, 16 threads per channel over the planes
__global__ void __launch_bounds__(256)
channel_planes_kernel(const float* __restrict__ planes, float* __restrict__ first, float* __restrict__ second, int channels, int splits,
                      float count, int statistics) {
  __shared__ float meet[2][256];
  const int tid = threadIdx.x, lane = tid & 15, row = tid >> 4, c = blockIdx.x * 16 + lane;
  float q[2][4] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
  if (c < channels) {
    int i = row;
    // sixteen loads in flight; with twice as many the conv_train step of [32][56][56][64] fp16 takes 151 us instead of 139
#pragma unroll 2
    for (; i + 48 < splits; i += 64) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        q[0][u] += planes[(int64_t)(2 * (i + 16 * u)) * channels + c];
        q[1][u] += planes[(int64_t)(2 * (i + 16 * u) + 1) * channels + c];
      }
    }
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      if (i + 16 * u >= splits) continue;
      q[0][u] += planes[(int64_t)(2 * (i + 16 * u)) * channels + c];
      q[1][u] += planes[(int64_t)(2 * (i + 16 * u) + 1) * channels + c];
    }
  }
#pragma unroll
  for (int w = 0; w < 2; ++w) meet[w][tid] = (q[w][0] + q[w][1]) + (q[w][2] + q[w][3]);
  __syncthreads();
  if (row > 0 || c >= channels) return;
#pragma unroll
  for (int w = 0; w < 2; ++w) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      q[w][u] = (meet[w][(4 * u) * 16 + lane] + meet[w][(4 * u + 1) * 16 + lane]) + (meet[w][(4 * u + 2) * 16 + lane] + meet[w][(4 * u + 3) * 16 + lane]);
  }
  float s = (q[0][0] + q[0][1]) + (q[0][2] + q[0][3]), t = (q[1][0] + q[1][1]) + (q[1][2] + q[1][3]);
  if (statistics) Statistics(count, &s, &t);
  first[c]  = s;
  second[c] = t;
}

// y = (x - mean) * rsqrt(variance + epsilon) * scale + bias, relu or not (GRAD = false), or the gradient
// scale * rsqrt(variance + epsilon) / count * (count * dy - sum_dy - (x - mean) * sum_dyx / (variance + epsilon)).
// A thread stays on its channels and walks pixels, so what depends on the channel alone is computed once per thread.
struct ApplyParams {
  const void *a, *x, *out;  // a: dy (GRAD only)
  const float *mean, *variance, *scale, *bias, *sum_dy, *sum_dyx;
  void* result;
  int64_t pixels;
  int channels, chunk_lanes, pixels_per_block, relu;
  float epsilon, count;
};

template <typename T, int E, bool GRAD, bool MASKED>
__global__ void __launch_bounds__(256)
channel_apply_kernel(ApplyParams p) {
  const int lanes = p.chunk_lanes, rows = 256 / lanes;
  const int ch = (blockIdx.x * lanes + threadIdx.x % lanes) * E;
  if (ch >= p.channels) return;
  const int64_t first = (int64_t)blockIdx.y * p.pixels_per_block;
  const int64_t end   = min(first + p.pixels_per_block, p.pixels);
  const T *a = static_cast<const T*>(p.a), *x = static_cast<const T*>(p.x), *o = static_cast<const T*>(p.out);
  T* result = static_cast<T*>(p.result);
  float mean[E], k0[E], k1[E], k2[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const float spread = p.variance[ch + e] + p.epsilon, inv = 1.0f / sqrtf(spread);
    mean[e] = p.mean[ch + e];
    if constexpr (GRAD) {
      k0[e] = p.scale[ch + e] * inv / p.count;
      k1[e] = p.sum_dy[ch + e];
      k2[e] = p.sum_dyx[ch + e] / spread;
    } else {
      k0[e] = inv;
      k1[e] = p.scale[ch + e];
      k2[e] = p.bias[ch + e];
    }
  }
  auto apply = [&](const float (&av)[E], const float (&xv)[E], const float (&ov)[E], int64_t at) {
    T r[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const float centred = xv[e] - mean[e];
      if constexpr (GRAD) {
        const float d = MASKED ? (ov[e] > 0.0f ? av[e] : 0.0f) : av[e];
        r[e]          = (T)(k0[e] * ((d * p.count - k1[e]) - centred * k2[e]));
      } else {
        const float y = centred * k0[e] * k1[e] + k2[e];
        r[e]          = (T)(p.relu && !(y > 0.0f) ? 0.0f : y);
      }
    }
    __builtin_memcpy(__builtin_assume_aligned(result + at, E * sizeof(T)), r, sizeof(r));
  };
  auto load = [&](float (&av)[E], float (&xv)[E], float (&ov)[E], int64_t at) {
    if (GRAD) LoadChannels<T, E>(a + at, av);
    LoadChannels<T, E>(x + at, xv);
    if (MASKED) LoadChannels<T, E>(o + at, ov);
  };
  int64_t q = first + threadIdx.x / lanes;
  for (; q + rows < end; q += 2 * rows) {
    float av[2][E], xv[2][E], ov[2][E];
#pragma unroll
    for (int u = 0; u < 2; ++u) load(av[u], xv[u], ov[u], (q + u * rows) * p.channels + ch);
#pragma unroll
    for (int u = 0; u < 2; ++u) apply(av[u], xv[u], ov[u], (q + u * rows) * p.channels + ch);
  }
  if (q < end) {
    float av[E], xv[E], ov[E];
    load(av, xv, ov, q * p.channels + ch);
    apply(av, xv, ov, q * p.channels + ch);
  }
}

// Channels of a thread: 16 bytes where the tensors allow it, and 4 where that would not give 256 CUs a block each at two pixels a
// thread.  Blocks by themselves on a CU are bound by one thread's instructions (eight channels' conversions, divisions and
// square roots, one after the other), not by loads: 525 pixels of 48 channels in fp16 took, sums 3.9, normalisation
// 4.2, gradient's sums 4.8, gradient 5.7 us with 2 to 4 blocks of wide threads, and 3.0, 3.6, 3.2 and 3.1 with 16 to 31 of
// narrow ones.  A line four times as high changes nothing for these kernels (60 convolutions' training steps: within 0.1% in the
// geometric mean), one a quarter as high loses 0.4%.
bool Few(int64_t pixels, int channels, int chunk) { return pixels * (channels / chunk) < 256 * 512; }

// lanes of a block side by side over channel chunks: a power of two, at most 64
int ChunkLanes(int chunks) {
  int lanes = 1;
  while (lanes < chunks && lanes < 64) lanes *= 2;
  return lanes;
}

template <typename T>
void Apply(ApplyParams p, bool grad, hipStream_t stream) {
  constexpr int E = 16 / (int)sizeof(T);
  auto aligned    = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; };
  const bool wide  = p.channels % E == 0 && aligned(p.a) && aligned(p.x) && aligned(p.out) && aligned(p.result);
  constexpr int F  = 4 / (int)sizeof(T);
  const bool few   = wide && Few(p.pixels, p.channels, E);
  const int chunks = p.channels / (few ? F : wide ? E : 1);
  p.chunk_lanes    = ChunkLanes(chunks);
  const int column_blocks = (chunks + p.chunk_lanes - 1) / p.chunk_lanes, rows = 256 / p.chunk_lanes;
  // four pixels per thread, more where that would be over 4096 blocks; two, one trip to memory, up to two blocks for every CU
  int64_t blocks = std::min<int64_t>(4096 / column_blocks, p.pixels / (4 * rows));
  blocks         = std::max<int64_t>({1, blocks, std::min<int64_t>(512 / column_blocks, p.pixels / (2 * rows))});
  p.pixels_per_block = (int)((p.pixels + blocks - 1) / blocks);
  blocks             = (p.pixels + p.pixels_per_block - 1) / p.pixels_per_block;
  const dim3 grid(column_blocks, (unsigned)blocks);
#define CINN_APPLY(E, GRAD, MASKED) hipLaunchKernelGGL((channel_apply_kernel<T, E, GRAD, MASKED>), grid, dim3(256), 0, stream, p)
  if (!grad) {
    if (few) CINN_APPLY(F, false, false);
    else if (wide) CINN_APPLY(E, false, false);
    else CINN_APPLY(1, false, false);
  } else if (p.out) {
    if (few) CINN_APPLY(F, true, true);
    else if (wide) CINN_APPLY(E, true, true);
    else CINN_APPLY(1, true, true);
  } else {
    if (few) CINN_APPLY(F, true, false);
    else if (wide) CINN_APPLY(E, true, false);
    else CINN_APPLY(1, true, false);
  }
#undef CINN_APPLY
  CINN_HIP_CALL(hipGetLastError());
}

template <typename T, int E, bool DIRECT>
void LaunchSums(const SumsParams& p, dim3 grid, bool grad, hipStream_t stream) {
  if (!grad) {
    hipLaunchKernelGGL((channel_sums_kernel<T, E, false, false, DIRECT>), grid, dim3(256), 0, stream, p);
  } else if (p.out) {
    hipLaunchKernelGGL((channel_sums_kernel<T, E, true, true, DIRECT>), grid, dim3(256), 0, stream, p);
  } else {
    hipLaunchKernelGGL((channel_sums_kernel<T, E, true, false, DIRECT>), grid, dim3(256), 0, stream, p);
  }
}

template <typename T>
void Sums(SumsParams p, bool grad, float* first, float* second, hipStream_t stream) {
  constexpr int E = 16 / (int)sizeof(T);
  auto aligned    = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; };
  const bool wide = p.channels % E == 0 && aligned(p.a) && aligned(p.x) && aligned(p.out);
  constexpr int F = 4 / (int)sizeof(T);
  bool few        = wide && Few(p.pixels, p.channels, E);
  int chunks      = p.channels / (few ? F : wide ? E : 1);
  p.chunk_lanes    = ChunkLanes(chunks);
  const int column_blocks = (chunks + p.chunk_lanes - 1) / p.chunk_lanes;
  const int rows          = 256 / p.chunk_lanes;
  // Two blocks for every CU, at least eight pixels for every thread; or as many as it loads at a time, one trip to memory, while
  // there are no more planes than channel_planes_kernel loads at a time (with two trips and more 5.5 us instead of 4.2 for the
  // gradient's sums of 3915 pixels of 16 channels in fp32).
  int64_t splits = std::min<int64_t>(512 / column_blocks, p.pixels / (8 * rows));
  splits = std::max<int64_t>({1, splits, std::min<int64_t>({64, 512 / column_blocks, p.pixels / ((grad ? 2 : 4) * rows)})});
  p.pixels_per_split = (int)((p.pixels + splits - 1) / splits);
  splits             = (p.pixels + p.pixels_per_split - 1) / p.pixels_per_split;
  p.splits = (int)splits, p.first = first, p.second = second;
  const size_t plane_bytes = (size_t)splits * 2 * p.channels * sizeof(float);
  dim3 grid(column_blocks, (unsigned)splits);
  if (plane_bytes > ScratchLimit(ScratchKind::kSplitK, stream)) {
    // under capture without an eager run or a reservation: a block walks all splits of its channels, four chunks of them,
    // and needs no planes
    few           = false;
    chunks        = p.channels / (wide ? E : 1);
    p.chunk_lanes = std::min(ChunkLanes(chunks), 4);
    grid          = dim3((chunks + p.chunk_lanes - 1) / p.chunk_lanes);
  } else {
    p.planes = static_cast<float*>(Scratch(ScratchKind::kSplitK, plane_bytes, stream));
  }
  if (!p.planes && wide) LaunchSums<T, E, true>(p, grid, grad, stream);
  if (!p.planes && !wide) LaunchSums<T, 1, true>(p, grid, grad, stream);
  if (p.planes && few) LaunchSums<T, F, false>(p, grid, grad, stream);
  if (p.planes && wide && !few) LaunchSums<T, E, false>(p, grid, grad, stream);
  if (p.planes && !wide) LaunchSums<T, 1, false>(p, grid, grad, stream);
  if (p.planes) {
    hipLaunchKernelGGL(channel_planes_kernel, dim3((p.channels + 15) / 16), dim3(256), 0, stream, p.planes, first, second, p.channels,
                       (int)splits, (float)p.pixels, grad ? 0 : 1);
  }
  CINN_HIP_CALL(hipGetLastError());
}

cinn_buffer_t* BufferArg(void* v_args, int index) {
  auto* args = static_cast<cinn_pod_value_t*>(v_args);
  CINN_RT_CHECK(args[index].type_code_ == CINN_POD_BUFFER_P, "channel call: argument %d is not a buffer", index);
  auto* b = static_cast<cinn_buffer_t*>(args[index].value_.v_handle);
  CINN_RT_CHECK(b && b->memory, "channel call: argument %d has no device memory", index);
  return b;
}
bool IsF32(const cinn_buffer_t* b) { return b->type.code == cinn_type_float && b->type.bits == 32; }
bool SameType(const cinn_buffer_t* a, const cinn_buffer_t* b) { return a->type.code == b->type.code && a->type.bits == b->type.bits; }
float* Vector(const cinn_buffer_t* b) {
  CINN_RT_CHECK(IsF32(b), "channel call: per-channel operands and results are fp32");
  return reinterpret_cast<float*>(b->memory);
}

// Arguments of a call with `outputs` results: operand slot s (four bits of `operands` each) says which input it is.
struct Operands {
  void* v_args;
  int inputs;
  unsigned long long slots;
  cinn_buffer_t* operator()(int slot) const {
    const int at = (int)((slots >> (4 * slot)) & 15);
    CINN_RT_CHECK(at < inputs, "channel call: operand %d is argument %d of %d inputs", slot, at, inputs);
    return BufferArg(v_args, at);
  }
};

void CheckExtents(int pixels, int channels) {
  CINN_RT_CHECK(pixels > 0 && channels > 0, "channel call: %d pixels of %d channels", pixels, channels);
}

// calls fn with a value of the element type
template <typename Fn>
void ByType(const cinn_buffer_t* b, Fn fn) {
  if (IsF32(b)) {
    fn(float());
  } else if (b->type.code == cinn_type_float && b->type.bits == 16) {
    fn(_Float16());
  } else {
    CINN_RT_CHECK(b->type.code == cinn_type_bfloat && b->type.bits == 16, "channel call: fp16 / bf16 / fp32 only");
    fn(__bf16());
  }
}

}  // namespace

extern "C" void cinn_call_hip_channel_statistics(void* v_args, int num_args, int pixels, int channels, void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  CINN_RT_CHECK(num_args == 3, "channel statistics: x, mean and variance expected, got %d arguments", num_args);
  CheckExtents(pixels, channels);
  const cinn_buffer_t* x = BufferArg(v_args, 0);
  SumsParams p{x->memory, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, pixels, channels, 0, 0, 0};
  float *mean = Vector(BufferArg(v_args, 1)), *variance = Vector(BufferArg(v_args, 2));
  ByType(x, [&](auto t) { Sums<decltype(t)>(p, false, mean, variance, static_cast<hipStream_t>(stream)); });
}

extern "C" void cinn_call_hip_channel_normalize(void* v_args, int num_args, int pixels, int channels, int operands, float epsilon,
                                                int relu, void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  CheckExtents(pixels, channels);
  const Operands in{v_args, num_args - 1, (unsigned)operands};
  const cinn_buffer_t *x = in(0), *y = BufferArg(v_args, num_args - 1);
  CINN_RT_CHECK(SameType(x, y), "channel normalize: x and y differ in type");
  ApplyParams p{};
  p.x = x->memory, p.result = y->memory, p.mean = Vector(in(1)), p.variance = Vector(in(2)), p.scale = Vector(in(3)), p.bias = Vector(in(4));
  p.pixels = pixels, p.channels = channels, p.relu = relu, p.epsilon = epsilon, p.count = (float)pixels;
  ByType(x, [&](auto t) { Apply<decltype(t)>(p, false, static_cast<hipStream_t>(stream)); });
}

extern "C" void cinn_call_hip_channel_gradient_sums(void* v_args, int num_args, int pixels, int channels, int operands, int masked,
                                                    void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  CheckExtents(pixels, channels);
  const Operands in{v_args, num_args - 2, (unsigned)operands};
  const cinn_buffer_t *dy = in(0), *x = in(1), *out = masked ? in(3) : nullptr;
  CINN_RT_CHECK(SameType(dy, x) && (!out || SameType(dy, out)), "channel gradient sums: operands of different types");
  SumsParams p{dy->memory, x->memory, out ? out->memory : nullptr, Vector(in(2)), nullptr, nullptr, nullptr, pixels, channels, 0, 0, 0};
  float *sum_dy = Vector(BufferArg(v_args, num_args - 2)), *sum_dyx = Vector(BufferArg(v_args, num_args - 1));
  ByType(dy, [&](auto t) { Sums<decltype(t)>(p, true, sum_dy, sum_dyx, static_cast<hipStream_t>(stream)); });
}

extern "C" void cinn_call_hip_channel_gradient(void* v_args, int num_args, int pixels, int channels, int operands, int masked,
                                               float epsilon, void* stream) {
  CINN_HIP_CLEAR_STALE_ERROR();
  CheckExtents(pixels, channels);
  const Operands in{v_args, num_args - 1, (unsigned)operands};
  const cinn_buffer_t *dy = in(0), *x = in(1), *out = masked ? in(7) : nullptr, *dx = BufferArg(v_args, num_args - 1);
  CINN_RT_CHECK(SameType(dy, x) && SameType(dy, dx) && (!out || SameType(dy, out)), "channel gradient: operands of different types");
  ApplyParams p{};
  p.a = dy->memory, p.x = x->memory, p.out = out ? out->memory : nullptr, p.result = dx->memory;
  p.mean = Vector(in(2)), p.variance = Vector(in(3)), p.scale = Vector(in(4)), p.sum_dy = Vector(in(5)), p.sum_dyx = Vector(in(6));
  p.pixels = pixels, p.channels = channels, p.epsilon = epsilon, p.count = (float)pixels;
  ByType(dy, [&](auto t) { Apply<decltype(t)>(p, true, static_cast<hipStream_t>(stream)); });
}
