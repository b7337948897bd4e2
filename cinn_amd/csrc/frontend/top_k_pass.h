// Selecting the first entries of a sorted axis without sorting (or storing) all of it.
//
// NetBuilder::TopK composes sort, argsort, two slices and a cast, as the reference does
// (cinn/frontend/decomposer/top_k.cc:22-47): two full sorts of the operand and two full-size results of which k entries
// are read.  This pass finds slice(sort(x)) and cast<int64>(slice(argsort(x).indices)) over the first k entries of the
// sorted axis, where nothing else reads the full results, and makes one hip_top_k instruction of the ones that share x,
// axis, direction and k.
#pragma once
#include <set>
#include <string>

#include "frontend/syntax.h"

namespace cinn {
namespace frontend {

Program FuseTopK(const Program& program, const std::set<std::string>& fetch_ids);

}  // namespace frontend
}  // namespace cinn
