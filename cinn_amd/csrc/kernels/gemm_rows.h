// Internal interface of the kernel for products of few rows (gemm_rows.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace cinn_hip_kernels {

// C [m][n] = act( norm(A) [m][k] . B^T * scale + shift + residual_scale * residual ), B stored [n][k], fp16 or bf16 (all
// matrices), m <= 64, k % 32 == 0.
struct RowProduct {
  bool bf16;
  const void* a;
  const void* b;
  void* c[3];          // n / width tensors [m][width], which take as many columns each
  int width;
  int m, n, k;
  const float* scale;  // per column, or null: alpha
  const float* shift;  // per column, or null
  float alpha;
  const void* residual;  // [m][n], or null; one result tensor then
  float residual_scale;
  bool relu, gelu;
  // layer norm of A's rows before the product: (x - mean) / sqrt(variance + epsilon) * gamma + beta, rounded to the type;
  // gamma and beta [k] of the matrices' type, null: none
  const void* gamma;
  const void* beta;
  float epsilon;
};

// longest row that is normalised: a lane holds 16 bytes of x, W, gamma and beta for each of its wavefront's five blocks of K (114
// registers; above 128 a CU holds one block)
constexpr int kRowProductMaxNormK = 1280;

// false where the kernel does not take the extents; operands lie at any address of their type
bool RowProductSupported(const RowProduct& p);
// which of the file's two kernels runs it: gemm_rows_ring_kernel (but for some single rows), or gemm_rows_kernel; by the addresses as
// well where there are any
bool RowRingTakes(const RowProduct& p);
// whether the kernel (`ring`: which one, as above) is ahead of the tiled ones for a product that it takes; `saves_launch`: several results, which would
// be copied out of one; `splits`: without a scale, which gemm_flex.hip would take and split its K
bool RowProductPays(int m, int n, int k, bool ring, bool saves_launch, bool splits);
// which of a layer norm before the product and a gelu behind it (those that there are) are faster inside
struct RowFusion {
  bool norm, gelu;
};
RowFusion ChooseRowFusion(int m, int n, int k, bool ring, RowFusion there);
void RunRowProduct(const RowProduct& p, hipStream_t stream);

}  // namespace cinn_hip_kernels
