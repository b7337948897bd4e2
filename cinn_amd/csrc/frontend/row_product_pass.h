// Products of few rows with what surrounds them in a decoding step.
#pragma once
#include <set>
#include <string>

#include "frontend/syntax.h"

namespace cinn {
namespace frontend {

// A linear layer of at most 64 rows (what FuseMatmulBias makes of a product with a const weight and bias) becomes one
// hip_matmul_rows with
//   * the layer norm of its rows, where the product alone reads it (PaddleLayerNorm's composition, scale and bias in the
//     element type),
//   * the gelu that alone reads it, on the fp32 sum,
//   * one result tensor for each of two or three slices that divide its columns.  Transposes behind them that only move an
//     axis of one become reshapes, which are no kernel.
// Each where the kernel is faster with it than without (gemm_rows.hip).  Layers with none of these keep their call in a program
// without any.  FLAGS_cinn_hip_gemm_skinny=0 leaves the program as it is.
Program FuseRowProducts(const Program& program, const std::set<std::string>& fetch_ids);

}  // namespace frontend
}  // namespace cinn
