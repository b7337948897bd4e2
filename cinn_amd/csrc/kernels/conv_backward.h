// Internal interface of the matrix-core convolution gradients (conv_backward_mfma.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "cinn_hip_runtime.h"

namespace cinn_hip_kernels {

struct ConvBackwardArgs {
  const void* x;   // input (filter gradient)
  const void* w;   // filter (data gradient)
  const void* dy;  // gradient of the output
  void* out;       // dx or dw: out = alpha * gradient + beta * out
  bool nhwc;       // else NCHW tensors and [F][C][KH][KW] filters
  int n, c, h, w_in;     // input extents
  int f, kh, kw;         // filter: f output channels
  int oh, ow;
  int pad_h, pad_w, stride_h, stride_w, dil_h, dil_w;
  float alpha, beta;
  cinn_type_t type;
};

// false when the shape or type is not theirs (fp64, extents beyond 32-bit offsets, empty ones, negative paddings, dilation
// together with a stride), or when the stream is being captured and its scratch is too small; groups are not supported
bool TryConvBackwardData(const ConvBackwardArgs& a, hipStream_t stream);
bool TryConvBackwardFilter(const ConvBackwardArgs& a, hipStream_t stream);

}  // namespace cinn_hip_kernels
