#include "frontend/attention_pass.h"

#include <algorithm>
#include <climits>
#include <map>
#include <vector>

#include "hlir/op.h"

namespace cinn {
namespace frontend {

namespace {

using hlir::framework::GetAttr;

// the operand slots of the call: q, the two pieces of k, the two pieces of v, the result
constexpr int kResult = 5;

// where an operand's rows lie: 0 = [b][h][t][d], 1 = [b][t][h][d]
struct Operand {
  Variable var;
  int layout{0};
};

bool SplitsHeads(const Instruction& ins) {
  return ins->op_type == "transpose" && ins->inputs.size() == 1 && ins->inputs[0]->shape.size() == 4 &&
         GetAttr<std::vector<int>>(ins->attrs, "axis", {}) == std::vector<int>{0, 2, 1, 3};
}

}  // namespace

Program FuseAttention(const Program& program, const std::set<std::string>& fetch_ids) {
  const auto& instrs = program.instructions();
  std::map<std::string, std::vector<size_t>> users;
  std::map<std::string, size_t> defined_at;
  for (size_t i = 0; i < instrs.size(); ++i) {
    for (auto& in : instrs[i]->inputs) users[in->id].push_back(i);
    for (auto& o : instrs[i]->outputs) defined_at[o->id] = i;
  }
  auto single_user = [&](const Variable& v) -> int {
    auto it = users.find(v->id);
    return fetch_ids.count(v->id) || it == users.end() || it->second.size() != 1 ? -1 : static_cast<int>(it->second[0]);
  };
  auto source = [&](const Variable& v) -> const Instruction* {
    auto it = defined_at.find(v->id);
    return it == defined_at.end() ? nullptr : &instrs[it->second];
  };
  auto in_place = [&](const Variable& v) {
    const Instruction* def = source(v);
    return def && SplitsHeads(*def) ? Operand{(*def)->inputs[0], 1} : Operand{v, 0};
  };
  // v, or the two pieces it is joined from along its rows
  auto pieces = [&](const Variable& v) {
    const Instruction* def = source(v);
    if (def && (*def)->op_type == "concat" && (*def)->inputs.size() == 2) {
      const int rank = static_cast<int>(v->shape.size());
      int axis       = GetAttr<int>((*def)->attrs, "axis", 0);
      if (axis < 0) axis += rank;
      if (axis == rank - 2 && (*def)->inputs[0]->type == v->type && (*def)->inputs[1]->type == v->type)
        return std::vector<Operand>{in_place((*def)->inputs[0]), in_place((*def)->inputs[1])};
    }
    return std::vector<Operand>{in_place(v)};
  };
  auto rows = [](const Operand& o) {
    const auto& s = o.var->shape;
    return o.layout == 0 ? s[s.size() - 2] : s[s.size() - 3];
  };

  std::vector<bool> dropped(instrs.size(), false);
  std::map<size_t, Instruction> replacement;
  for (size_t i = 0; i < instrs.size(); ++i) {
    const auto& qk = instrs[i];
    if (qk->op_type != "matmul" || qk->inputs.size() != 2 || GetAttr<bool>(qk->attrs, "trans_a", false) ||
        !GetAttr<bool>(qk->attrs, "trans_b", false))
      continue;
    const Variable &q = qk->inputs[0], &k = qk->inputs[1];
    const int rank = static_cast<int>(q->shape.size());
    if ((rank != 3 && rank != 4) || k->shape.size() != q->shape.size() || !(q->type == k->type)) continue;
    if (!q->type.is_float(32) && !q->type.is_float(16) && !q->type.is_bfloat16()) continue;
    const int softmax_at = single_user(qk->outputs[0]);
    if (softmax_at < 0 || instrs[softmax_at]->op_type != "softmax") continue;
    const auto axes = GetAttr<std::vector<int>>(instrs[softmax_at]->attrs, "axes", {-1});
    if (axes.size() != 1 || (axes[0] != -1 && axes[0] != rank - 1)) continue;
    const int pv_at = single_user(instrs[softmax_at]->outputs[0]);
    if (pv_at < 0) continue;
    const auto& pv = instrs[pv_at];
    if (pv->op_type != "matmul" || pv->inputs.size() != 2 || !(pv->inputs[0] == instrs[softmax_at]->outputs[0]) ||
        GetAttr<bool>(pv->attrs, "trans_a", false) || GetAttr<bool>(pv->attrs, "trans_b", false) ||
        GetAttr<float>(pv->attrs, "alpha", 1.0f) != 1.0f)
      continue;
    const Variable& v = pv->inputs[1];
    // the same batch entries and row length throughout
    const int d = q->shape[rank - 1], queries = q->shape[rank - 2], keys = k->shape[rank - 2];
    if (v->shape != k->shape || !(v->type == q->type) || k->shape[rank - 1] != d || keys < 1 || queries < 1) continue;
    if (!std::equal(q->shape.begin(), q->shape.end() - 2, k->shape.begin())) continue;
    if (d > 128 || d % (16 / q->type.bytes()) != 0) continue;
    const int batch = q->shape[0], heads = rank == 4 ? q->shape[1] : 1;
    if (static_cast<int64_t>(batch) * heads * queries >= INT_MAX ||
        static_cast<int64_t>(batch) * heads * d * std::max(queries, keys) >= INT_MAX)
      continue;

    auto ks = pieces(k), vs = pieces(v);
    // pieces that do not correspond: the joined tensors
    if (ks.size() != vs.size() || rows(ks[0]) != rows(vs[0])) ks = {in_place(k)}, vs = {in_place(v)};
    Operand slots[kResult + 1];
    slots[0] = in_place(q);
    for (size_t j = 0; j < ks.size(); ++j) slots[1 + j] = ks[j], slots[3 + j] = vs[j];
    slots[kResult] = {pv->outputs[0], 0};
    const int merge_at = rank == 4 ? single_user(pv->outputs[0]) : -1;
    if (merge_at >= 0 && SplitsHeads(instrs[merge_at])) {
      slots[kResult]    = {instrs[merge_at]->outputs[0], 1};
      dropped[merge_at] = true;
    }

    Instruction call("hip_attention");
    int operands = 0, layouts = 0;
    for (int s = 0; s <= kResult; ++s) {
      if (!slots[s].var.defined()) continue;
      layouts |= slots[s].layout << (4 * s);
      if (s == kResult) break;
      auto& in = call->inputs;
      auto at  = std::find(in.begin(), in.end(), slots[s].var);
      operands |= static_cast<int>(at - in.begin()) << (4 * s);
      if (at == in.end()) in.push_back(slots[s].var);
    }
    call->outputs = {slots[kResult].var};
    call->attrs   = {{"scale", GetAttr<float>(qk->attrs, "alpha", 1.0f)},
                     {"batch", batch},
                     {"heads", heads},
                     {"queries", queries},
                     {"keys", rows(ks[0])},
                     {"appended", ks.size() > 1 ? rows(ks[1]) : 0},
                     {"d", d},
                     {"operands", operands},
                     {"layouts", layouts},
                     {"out_shape", slots[kResult].var->shape}};
    replacement.emplace(pv_at, call);
    dropped[i] = dropped[softmax_at] = dropped[pv_at] = true;
  }
  if (replacement.empty()) return program;

  // transposes and concatenations that only the replaced products read
  std::map<std::string, int> readers;
  for (size_t i = 0; i < instrs.size(); ++i)
    if (!dropped[i])
      for (auto& in : instrs[i]->inputs) ++readers[in->id];
  for (auto& r : replacement)
    for (auto& in : r.second->inputs) ++readers[in->id];
  for (size_t i = instrs.size(); i-- > 0;) {
    const auto& ins = instrs[i];
    if (dropped[i] || !(SplitsHeads(ins) || ins->op_type == "concat")) continue;
    const auto& out = ins->outputs[0];
    if (readers[out->id] > 0 || fetch_ids.count(out->id) || !users.count(out->id)) continue;
    dropped[i] = true;
    for (auto& in : ins->inputs) --readers[in->id];
  }

  std::vector<Instruction> out;
  for (size_t i = 0; i < instrs.size(); ++i) {
    auto r = replacement.find(i);
    if (r != replacement.end()) {
      out.push_back(r->second);
    } else if (!dropped[i]) {
      out.push_back(instrs[i]);
    }
  }
  return Program(std::move(out), program.GetInputs(), program.name());
}

}  // namespace frontend
}  // namespace cinn
