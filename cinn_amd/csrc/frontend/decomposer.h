// Program pass that rewrites composite operators into the primitives the backend fuses.  It covers
// the two decompositions the GPU configs need:
//   softmax     cinn/frontend/decomposer/activation.cc:70-118 (mode "fast": exp(x) / sum(exp(x));
//               any other mode subtracts the row maximum first)
//   batch_norm  inference form with the operation order of pe::BatchNorm_NCHW
//               (cinn/hlir/pe/nn.cc:700-721): (x - mean) * scale / sqrt(variance + eps) + bias
//   batch_norm_train / batch_norm_grad  on channels-last tensors the calls of kernels/channel_sums.hip, a relu after the
//               first and the relu_grad before the second taken along; else primitives
#pragma once
#include <map>
#include <set>
#include <string>

#include "frontend/syntax.h"

namespace cinn {
namespace frontend {

// Returns the rewritten program.  Output variables of rewritten instructions keep their ids; `fetch_ids` are the values a
// caller reads.
Program ApplyDecomposer(const Program& program, const std::set<std::string>& fetch_ids = {});

}  // namespace frontend
}  // namespace cinn
