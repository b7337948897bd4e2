// Attention as one instruction.
//
// softmax(matmul(q, k, transposed, alpha)) over the last axis, multiplied by v, becomes hip_attention where nothing else
// reads scores or probabilities.  The call reads every operand where its producer left it, so that the transposes which
// split heads off a projection ([b][t][h][d] -> [b][h][t][d]), the one that merges them again, and the concatenations
// which append new keys and values to a cache go too, unless something else reads them.  The scores and probabilities it
// does not store were rounded to the element type; here they stay fp32 up to the second product's operand.  The softmax
// subtracts the row's maximum in either mode, so that exponentials which overflow in mode "fast" do not.
#pragma once
#include <set>
#include <string>

#include "frontend/syntax.h"

namespace cinn {
namespace frontend {

// The three projections of one input that such an attention reads, x W + b with const W and b each, as one product with
// joined weights (joined before the first run): one launch of three times the columns, which fills the chip where one of
// them does not, instead of three.  Queries, keys and values are then parts of its rows, which hip_attention reads where
// they lie; whatever else reads a part gets a slice.  Runs after PretransposeConstMatmulWeights.
Program MergeProjections(const Program& program, const std::set<std::string>& fetch_ids);

Program FuseAttention(const Program& program, const std::set<std::string>& fetch_ids);

}  // namespace frontend
}  // namespace cinn
