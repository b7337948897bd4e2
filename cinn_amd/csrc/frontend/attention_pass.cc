#include "frontend/attention_pass.h"

#include <algorithm>
#include <climits>
#include <cmath>
#include <map>
#include <vector>

#include "frontend/pass_util.h"
#include "hlir/op.h"

namespace cinn {
namespace frontend {

namespace {

using hlir::framework::GetAttr;

// the operand slots of the call: q, the two pieces of k, the two pieces of v, the result
constexpr int kResult = 5;

// where an operand's rows lie: 0 = [b][h][t][d], 1 = [b][t][h][d], 2 + j = part j of [b][t][parts][h][d]
struct Operand {
  Variable var;
  int layout{0};
  int rows{0};
  int parts{1};
};

bool SplitsHeads(const Instruction& ins) {
  return ins->op_type == "transpose" && ins->inputs.size() == 1 && ins->inputs[0]->shape.size() == 4 &&
         GetAttr<std::vector<int>>(ins->attrs, "axis", {}) == std::vector<int>{0, 2, 1, 3};
}

// The matmul at qk, the softmax that alone reads it and the matmul that alone reads that, where hip_attention computes the
// same: fills in the positions of the other two.
bool IsAttention(const std::vector<Instruction>& instrs, const std::map<std::string, std::vector<size_t>>& users,
                 const std::set<std::string>& fetch_ids, const Instruction& qk, size_t* softmax_at, size_t* pv_at) {
  auto only_reader = [&](const Variable& v, size_t* at) {
    auto it = users.find(v->id);
    if (fetch_ids.count(v->id) || it == users.end() || it->second.size() != 1) return false;
    *at = it->second[0];
    return true;
  };
  if (qk->op_type != "matmul" || qk->inputs.size() != 2 || GetAttr<bool>(qk->attrs, "trans_a", false) ||
      !GetAttr<bool>(qk->attrs, "trans_b", false))
    return false;
  const Variable &q = qk->inputs[0], &k = qk->inputs[1];
  const int rank = static_cast<int>(q->shape.size());
  if ((rank != 3 && rank != 4) || k->shape.size() != q->shape.size() || !(q->type == k->type)) return false;
  if (!q->type.is_float(32) && !q->type.is_float(16) && !q->type.is_bfloat16()) return false;
  // 0 times a score that overflows is no number, nor is the softmax of infinite ones: left to the operators
  const float alpha = GetAttr<float>(qk->attrs, "alpha", 1.0f);
  if (alpha == 0.0f || !std::isfinite(alpha)) return false;
  if (!only_reader(qk->outputs[0], softmax_at) || instrs[*softmax_at]->op_type != "softmax") return false;
  const auto axes = GetAttr<std::vector<int>>(instrs[*softmax_at]->attrs, "axes", {-1});
  if (axes.size() != 1 || (axes[0] != -1 && axes[0] != rank - 1)) return false;
  if (!only_reader(instrs[*softmax_at]->outputs[0], pv_at)) return false;
  const auto& pv = instrs[*pv_at];
  if (pv->op_type != "matmul" || pv->inputs.size() != 2 || !(pv->inputs[0] == instrs[*softmax_at]->outputs[0]) ||
      GetAttr<bool>(pv->attrs, "trans_a", false) || GetAttr<bool>(pv->attrs, "trans_b", false) ||
      GetAttr<float>(pv->attrs, "alpha", 1.0f) != 1.0f)
    return false;
  // the same batch entries and row length throughout
  const Variable& v = pv->inputs[1];
  const int d = q->shape[rank - 1], queries = q->shape[rank - 2], keys = k->shape[rank - 2];
  if (v->shape != k->shape || !(v->type == q->type) || k->shape[rank - 1] != d || keys < 1 || queries < 1) return false;
  if (!std::equal(q->shape.begin(), q->shape.end() - 2, k->shape.begin())) return false;
  if (d > 128 || d % (16 / q->type.bytes()) != 0) return false;
  const int batch = q->shape[0], heads = rank == 4 ? q->shape[1] : 1;
  return static_cast<int64_t>(batch) * heads * queries < INT_MAX &&
         static_cast<int64_t>(batch) * heads * d * std::max(queries, keys) < INT_MAX;
}

// x W + b with a const 2-D W stored [N][K] (its transposition may stand before it) and a const b, split into heads
struct Projection {
  size_t matmul, broadcast, add;
  Variable x, weight, bias;
};

}  // namespace

Program MergeProjections(const Program& program, const std::set<std::string>& fetch_ids) {
  const auto& instrs = program.instructions();
  std::map<std::string, std::vector<size_t>> users;
  std::map<std::string, size_t> defined_at;
  for (size_t i = 0; i < instrs.size(); ++i) {
    for (auto& in : instrs[i]->inputs) users[in->id].push_back(i);
    for (auto& o : instrs[i]->outputs) defined_at[o->id] = i;
  }
  auto only_reader = [&](const Variable& v) -> const Instruction* {
    auto it = users.find(v->id);
    return fetch_ids.count(v->id) || it == users.end() || it->second.size() != 1 ? nullptr : &instrs[it->second[0]];
  };
  auto source = [&](const Variable& v) -> const Instruction* {
    auto it = defined_at.find(v->id);
    return it == defined_at.end() ? nullptr : &instrs[it->second];
  };
  // a value that exists before the program's first instruction: const, or the transposition of such a one
  auto hoistable = [&](const Variable& v) {
    const Instruction* def = source(v);
    return def ? (*def)->op_type == "transpose" && (*def)->inputs[0]->is_const && !source((*def)->inputs[0]) && !fetch_ids.count(v->id)
               : v->is_const;
  };
  // split heads [b][h][t][d] back to the projection they come from
  auto projection = [&](const Variable& heads, Projection* p) {
    const Instruction* split = source(heads);
    if (!split || !SplitsHeads(*split)) return false;
    const Variable& rows         = (*split)->inputs[0];
    const Instruction* reshape   = source(rows);
    if (!reshape || (*reshape)->op_type != "reshape" || !only_reader(rows)) return false;
    const Variable& sum = (*reshape)->inputs[0];
    const Instruction* add = source(sum);
    if (!add || (*add)->op_type != "elementwise_add" || (*add)->inputs.size() != 2 || sum->shape.size() != 2 || !only_reader(sum)) return false;
    for (int side = 0; side < 2; ++side) {
      const Variable &prod = (*add)->inputs[side], &wide = (*add)->inputs[1 - side];
      const Instruction *mm = source(prod), *bc = source(wide);
      if (!mm || !bc || (*mm)->op_type != "matmul" || (*bc)->op_type != "broadcast_to" || !only_reader(prod) || !only_reader(wide)) continue;
      if ((*mm)->inputs.size() != 2 || GetAttr<bool>((*mm)->attrs, "trans_a", false) || !GetAttr<bool>((*mm)->attrs, "trans_b", false) ||
          GetAttr<float>((*mm)->attrs, "alpha", 1.0f) != 1.0f)
        continue;
      const Variable &x = (*mm)->inputs[0], &w = (*mm)->inputs[1], &bias = (*bc)->inputs[0];
      if (x->shape.size() != 2 || w->shape.size() != 2 || prod->shape != sum->shape || wide->shape != sum->shape) continue;
      if (bias->shape != std::vector<int>{sum->shape[1]} || GetAttr<std::vector<int>>((*bc)->attrs, "broadcast_axes", {}) != std::vector<int>{1})
        continue;
      if (!hoistable(w) || !bias->is_const || source(bias) || !(w->type == x->type) || !(bias->type == x->type)) continue;
      if (sum->shape[1] != rows->shape[2] * rows->shape[3] || sum->shape[0] != rows->shape[0] * rows->shape[1]) continue;
      *p = Projection{defined_at[prod->id], defined_at[wide->id], defined_at[sum->id], x, w, bias};
      return true;
    }
    return false;
  };

  std::vector<bool> dropped(instrs.size(), false);
  std::map<size_t, std::vector<Instruction>> before;       // emitted in front of an instruction
  std::map<size_t, Instruction> replacement;
  int serial = 0;
  for (auto& qk : instrs) {
    size_t softmax_at, pv_at;
    if (!IsAttention(instrs, users, fetch_ids, qk, &softmax_at, &pv_at) || qk->inputs[0]->shape.size() != 4) continue;
    const Instruction& pv = instrs[pv_at];
    // what this program computes of keys and values: all of them, or what it appends to a cache
    auto computed = [&](const Variable& v) {
      const Instruction* def = source(v);
      return def && (*def)->op_type == "concat" && (*def)->inputs.size() == 2 ? (*def)->inputs[1] : v;
    };
    Projection p[3];
    if (!projection(qk->inputs[0], &p[0]) || !projection(computed(qk->inputs[1]), &p[1]) || !projection(computed(pv->inputs[1]), &p[2]))
      continue;
    bool alike = p[0].add != p[1].add && p[1].add != p[2].add && p[0].add != p[2].add;
    for (auto& q : p)
      alike = alike && q.x == p[0].x && q.weight->shape == p[0].weight->shape && q.weight->type == p[0].weight->type &&
              !dropped[q.matmul] && !dropped[q.add];
    if (!alike) continue;
    const int rows = p[0].x->shape[0], width = p[0].weight->shape[0];
    if (static_cast<int64_t>(rows) * width * 3 >= INT_MAX) continue;

    const size_t first = std::min({p[0].matmul, p[1].matmul, p[2].matmul});
    auto& seq          = before[first];
    std::vector<Variable> weights, biases;
    for (auto& q : p) {
      const Instruction* def = source(q.weight);
      if (def && defined_at[q.weight->id] > first && !dropped[defined_at[q.weight->id]]) {
        seq.push_back(*def);
        dropped[defined_at[q.weight->id]] = true;
      }
      weights.push_back(q.weight);
      biases.push_back(q.bias);
    }
    Emitter e(&seq, "qkv" + std::to_string(serial++) + "_");
    auto weight  = e.Emit1("concat", weights, {{"axis", 0}});
    auto bias    = e.Emit1("concat", biases, {{"axis", 0}});
    auto product = e.Emit1("matmul", {p[0].x, weight}, instrs[p[0].matmul]->attrs);
    auto wide    = e.Emit1("broadcast_to", {bias}, {{"out_shape", std::vector<int>{rows, 3 * width}}, {"broadcast_axes", std::vector<int>{1}}});
    auto sum     = e.Emit1("elementwise_add", {product, wide}, instrs[p[0].add]->attrs);
    for (int j = 0; j < 3; ++j) {
      Instruction part("slice");
      part->inputs  = {sum};
      part->outputs = instrs[p[j].add]->outputs;
      part->attrs   = {{"axes", std::vector<int>{1}},
                       {"starts", std::vector<int>{j * width}},
                       {"ends", std::vector<int>{(j + 1) * width}},
                       {"infer_flags", std::vector<int>{}},
                       {"strides", std::vector<int>{}},
                       {"decrease_axis", std::vector<int>{}}};
      replacement.emplace(p[j].add, part);
      dropped[p[j].matmul] = dropped[p[j].broadcast] = true;
    }
  }
  if (replacement.empty()) return program;
  std::vector<Instruction> out;
  for (size_t i = 0; i < instrs.size(); ++i) {
    auto b = before.find(i);
    if (b != before.end()) out.insert(out.end(), b->second.begin(), b->second.end());
    auto r = replacement.find(i);
    if (r != replacement.end()) {
      out.push_back(r->second);
    } else if (!dropped[i]) {
      out.push_back(instrs[i]);
    }
  }
  return Program(std::move(out), program.GetInputs(), program.name());
}

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
  std::vector<bool> dropped(instrs.size(), false);
  auto in_place = [&](const Variable& v) {
    const Instruction* def = source(v);
    // a transpose that an earlier attention's call has taken along has no operand left: that call writes v itself
    if (!def || !SplitsHeads(*def) || dropped[defined_at[v->id]]) return Operand{v, 0, v->shape[v->shape.size() - 2], 1};
    const Variable& split  = (*def)->inputs[0];
    const Operand own{split, 1, split->shape[1], 1};
    // one part of packed projections
    const Instruction* reshape = source(split);
    const Instruction* slice   = reshape && (*reshape)->op_type == "reshape" ? source((*reshape)->inputs[0]) : nullptr;
    if (!slice || (*slice)->op_type != "slice") return own;
    const Variable &packed = (*slice)->inputs[0], &part = (*slice)->outputs[0];
    auto attr = [&](const char* name) { return GetAttr<std::vector<int>>((*slice)->attrs, name, {}); };
    const int width = split->shape[2] * split->shape[3];
    if (packed->shape.size() != 2 || part->shape != std::vector<int>{split->shape[0] * split->shape[1], width} ||
        packed->shape[0] != part->shape[0] || attr("axes") != std::vector<int>{1} || attr("starts").size() != 1 || !attr("strides").empty())
      return own;
    const int start = attr("starts")[0], parts = packed->shape[1] / width;
    if (packed->shape[1] % width != 0 || start < 0 || start % width != 0 || parts > 8) return own;
    return Operand{packed, 2 + start / width, split->shape[1], parts};
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
  auto rows = [](const Operand& o) { return o.rows; };

  std::map<size_t, Instruction> replacement;
  for (size_t i = 0; i < instrs.size(); ++i) {
    const auto& qk = instrs[i];
    size_t softmax_at, pv_at;
    if (!IsAttention(instrs, users, fetch_ids, qk, &softmax_at, &pv_at)) continue;
    const auto& pv = instrs[pv_at];
    const Variable &q = qk->inputs[0], &k = qk->inputs[1], &v = pv->inputs[1];
    const int rank = static_cast<int>(q->shape.size());
    const int d = q->shape[rank - 1], queries = q->shape[rank - 2], keys = k->shape[rank - 2];
    const int batch = q->shape[0], heads = rank == 4 ? q->shape[1] : 1;

    auto ks = pieces(k), vs = pieces(v);
    // pieces that do not correspond: the joined tensors
    if (ks.size() != vs.size() || rows(ks[0]) != rows(vs[0])) ks = {in_place(k)}, vs = {in_place(v)};
    Operand slots[kResult + 1];
    slots[0] = in_place(q);
    for (size_t j = 0; j < ks.size(); ++j) slots[1 + j] = ks[j], slots[3 + j] = vs[j];
    slots[kResult] = Operand{pv->outputs[0], 0, queries, 1};
    const int merge_at = rank == 4 ? single_user(pv->outputs[0]) : -1;
    if (merge_at >= 0 && SplitsHeads(instrs[merge_at])) {
      slots[kResult]    = Operand{instrs[merge_at]->outputs[0], 1, queries, 1};
      dropped[merge_at] = true;
    }

    // one number of parts per call, and offsets into packed rows that fit; else the parts by themselves
    int parts = 1;
    for (auto& s : slots) parts = std::max(parts, s.var.defined() ? s.parts : 1);
    bool packed = static_cast<int64_t>(batch) * heads * d * std::max(queries, keys) * parts < INT_MAX;
    for (auto& s : slots) packed = packed && (!s.var.defined() || s.layout < 2 || s.parts == parts);
    if (!packed) {
      for (int s = 0; s < kResult; ++s) {
        if (slots[s].layout < 2) continue;
        const Variable& v = s == 0 ? q : s < 3 ? k : pv->inputs[1];
        const Instruction* joined = source(v);
        const bool two            = s > 0 && ks.size() > 1;
        const Variable& own       = two ? (*joined)->inputs[s == 2 || s == 4 ? 1 : 0] : v;
        slots[s]                  = Operand{(*source(own))->inputs[0], 1, slots[s].rows, 1};
      }
      parts = 1;
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
                     {"parts", parts},
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
    if (dropped[i] || !(SplitsHeads(ins) || ins->op_type == "concat" || ins->op_type == "reshape" || ins->op_type == "slice")) continue;
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
