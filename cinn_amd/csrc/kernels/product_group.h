// Matrix products that do not depend on each other, in one launch (gemm_mfma.hip, gemm_flex.hip).
#pragma once

namespace cinn_hip_kernels {

// While an object lives, the products that its thread requests (cinn_call_cublas, cinn_call_hip_matmul_bias) wait: for Run, or for
// one that reads or writes what a waiting one writes, writes what it reads, or is meant for another stream.  They are launched
// then, together where that is faster.  Nothing else that reads or writes their memory may be requested in between.
class ProductGroup {
 public:
  ProductGroup();
  ~ProductGroup();  // drops what still waits: an exception is on its way
  ProductGroup(const ProductGroup&) = delete;
  ProductGroup& operator=(const ProductGroup&) = delete;
  void Run();
};

}  // namespace cinn_hip_kernels
