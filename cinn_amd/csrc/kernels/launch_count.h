// Which kernels a dispatch has chosen: counters of launches in this process.  For tests, which compare values and would not
// notice that another kernel computed them; nothing reads them to decide anything.
#pragma once
#include <atomic>

namespace cinn_hip_kernels {

enum Counted : int {
  kCountConvFew = 0,  // conv_few_kernel, one for each of its five tiles
  kCountConvPatch = 5,
  kCountRowsRing,
  kCountRows,
  kCountProductGroup,
  kCounted,
};
extern std::atomic<long long> g_launches[kCounted];  // conv_few_mfma.hip

inline void CountLaunch(int which) { g_launches[which].fetch_add(1, std::memory_order_relaxed); }

}  // namespace cinn_hip_kernels

// launches of `which` so far, -1 if there is no such counter; exported, deliberately absent from the public header
extern "C" long long cinn_hip_launches(int which);
