#include "frontend/top_k_pass.h"

#include <map>
#include <tuple>
#include <vector>

#include "frontend/pass_util.h"
#include "hlir/op.h"

namespace cinn {
namespace frontend {

namespace {

using hlir::framework::GetAttr;

int AxisOf(const Instruction& sort) {
  int axis = GetAttr<int>(sort->attrs, "axis", 0);
  return axis < 0 ? axis + static_cast<int>(sort->inputs[0]->shape.size()) : axis;
}

// the first k entries along `axis`, nothing else cut or dropped: k, else 0
int LeadingEntries(const Instruction& slice, int axis) {
  auto axes    = GetAttr<std::vector<int>>(slice->attrs, "axes", {});
  auto starts  = GetAttr<std::vector<int>>(slice->attrs, "starts", {});
  auto strides = GetAttr<std::vector<int>>(slice->attrs, "strides", {});
  const auto& in  = slice->inputs[0]->shape;
  const auto& out = slice->outputs[0]->shape;
  if (axes.size() != 1 || starts.size() != 1 || starts[0] != 0 || out.size() != in.size()) return 0;
  if (!strides.empty() && strides[0] != 1) return 0;
  if ((axes[0] < 0 ? axes[0] + static_cast<int>(in.size()) : axes[0]) != axis) return 0;
  return out[axis];
}

}  // namespace

Program FuseTopK(const Program& program, const std::set<std::string>& fetch_ids) {
  const auto& instrs = program.instructions();
  std::map<std::string, std::vector<size_t>> users;
  for (size_t i = 0; i < instrs.size(); ++i)
    for (auto& in : instrs[i]->inputs) users[in->id].push_back(i);
  auto single_user = [&](const Variable& v) -> int {
    auto it = users.find(v->id);
    return fetch_ids.count(v->id) || it == users.end() || it->second.size() != 1 ? -1 : static_cast<int>(it->second[0]);
  };
  auto unused = [&](const Variable& v) { return !fetch_ids.count(v->id) && !users.count(v->id); };

  struct Match {
    Variable values, indices;  // undefined when the program has only the other one
    size_t first;              // position of the earlier sort: x exists there
  };
  std::map<std::tuple<std::string, int, bool, int>, Match> matches;  // x, axis, ascending, k
  std::vector<bool> dropped(instrs.size(), false);
  for (size_t i = 0; i < instrs.size(); ++i) {
    const auto& sort = instrs[i];
    const bool values = sort->op_type == "sort", indices = sort->op_type == "argsort";
    if (!values && !indices) continue;
    const auto& type = sort->inputs[0]->type;
    if (!type.is_float(32) && !type.is_float(16) && !type.is_bfloat16() && !type.is_int(32)) continue;
    const int axis = AxisOf(sort);
    if (sort->inputs[0]->shape[axis] > 16384) continue;  // one block's LDS
    if (indices && !unused(sort->outputs[1])) continue;  // the positions are wanted
    const int slice_at = single_user(sort->outputs[0]);
    if (slice_at < 0 || instrs[slice_at]->op_type != "slice") continue;
    const int k = LeadingEntries(instrs[slice_at], axis);
    if (k <= 0) continue;
    Variable result = instrs[slice_at]->outputs[0];
    int cast_at     = -1;
    if (indices) {
      cast_at = single_user(result);
      if (cast_at < 0 || instrs[cast_at]->op_type != "cast" || !instrs[cast_at]->outputs[0]->type.is_int(64)) continue;
      result = instrs[cast_at]->outputs[0];
    }
    auto& m = matches.emplace(std::make_tuple(sort->inputs[0]->id, axis, GetAttr<bool>(sort->attrs, "is_ascend", true), k),
                              Match{Variable(), Variable(), i}).first->second;
    if (values ? m.values.defined() : m.indices.defined()) continue;  // a second one of the same kind stays as it is
    (values ? m.values : m.indices) = result;
    dropped[i] = dropped[slice_at] = true;
    if (cast_at >= 0) dropped[cast_at] = true;
  }
  if (matches.empty()) return program;

  std::vector<Instruction> out;
  for (size_t i = 0; i < instrs.size(); ++i) {
    for (auto& entry : matches) {
      const Match& m = entry.second;
      if (m.first != i || (!m.values.defined() && !m.indices.defined())) continue;
      Instruction top("hip_top_k");
      top->inputs  = {instrs[i]->inputs[0]};
      top->attrs   = {{"axis", std::get<1>(entry.first)},
                      {"is_ascend", std::get<2>(entry.first)},
                      {"k", std::get<3>(entry.first)},
                      {"outputs", (m.values.defined() ? 1 : 0) + (m.indices.defined() ? 2 : 0)}};
      if (m.values.defined()) top->outputs.push_back(m.values);
      if (m.indices.defined()) top->outputs.push_back(m.indices);
      out.push_back(top);
    }
    if (!dropped[i]) out.push_back(instrs[i]);
  }
  return Program(std::move(out), program.GetInputs(), program.name());
}

}  // namespace frontend
}  // namespace cinn
