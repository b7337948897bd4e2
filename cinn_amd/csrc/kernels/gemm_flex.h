// Internal interface of the register-staged MFMA kernel for products of any extents and layouts (gemm_flex.hip): the
// matrix products the direct-to-LDS kernels of gemm_mfma.hip do not take.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace cinn_hip_kernels {

enum class FlexType : int { kF16, kBF16, kF32 };

// C[m][n] = acc * alpha + shift[n] + residual_scale * residual[m][n], acc = sum_k A[m][k] B[k][n]
struct FlexGemm {
  FlexType type;
  const void* a;  // [m][k] when a_kc, else [k][m]; row pitch lda elements
  const void* b;  // [n][k] when b_kc, else [k][n]; row pitch ldb elements
  void* c;        // [m][n], row pitch n
  int m, n, k;
  bool a_kc, b_kc;
  int64_t lda, ldb;
  int batch = 1;
  int64_t stride_a = 0, stride_b = 0, stride_c = 0;  // elements between batch entries; 0 shares the operand
  const float* shift    = nullptr;
  const void* shift16   = nullptr;  // the shift in the matrices' 16-bit type
  const void* residual  = nullptr;  // of C's shape and batch stride
  float alpha           = 1.0f;
  float residual_scale  = 0.0f;
};

// block tile, groups of wavefronts and K split, and the estimate (microseconds) they were chosen by
struct FlexPlan {
  int tile, kg, splits;
  double us;
};

// false when an extent is beyond the kernel's 32-bit tile offsets (the caller then has a slower form)
bool PlanFlexGemm(const FlexGemm& g, hipStream_t stream, FlexPlan* plan);
void RunFlexGemm(const FlexGemm& g, FlexPlan plan, hipStream_t stream);

// Up to kFlexGroup unbatched products of one type in one launch; `alone` is how each would run by itself.  false when that is
// estimated to be faster.
constexpr int kFlexGroup = 4;
bool TryFlexGroup(const FlexGemm* g, const FlexPlan* alone, int count, hipStream_t stream);

}  // namespace cinn_hip_kernels
