#include "frontend/row_product_pass.h"

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <map>
#include <vector>

#include "frontend/pass_util.h"
#include "hlir/op.h"
#include "kernels/gemm_rows.h"

namespace cinn {
namespace frontend {

namespace {

using hlir::framework::GetAttr;
using utils::ShapeType;

class RowProductFuser {
 public:
  RowProductFuser(const Program& program, const std::set<std::string>& fetch_ids)
      : program_(program), fetch_ids_(fetch_ids), instrs_(program.instructions()), dropped_(instrs_.size(), false) {
    for (size_t i = 0; i < instrs_.size(); ++i) {
      for (auto& in : instrs_[i]->inputs) users_[in->id].push_back(i);
      for (auto& o : instrs_[i]->outputs) defined_at_[o->id] = i;
    }
  }

  Program Run() {
    for (size_t i = 0; i < instrs_.size(); ++i)
      if (instrs_[i]->op_type == "hip_conv2d_bn_relu") Fuse(i, false);
    if (replacement_.empty()) return program_;
    // the other layers between them: as images they would leave reshapes of two readers, which are copies
    for (size_t i = 0; i < instrs_.size(); ++i)
      if (instrs_[i]->op_type == "hip_conv2d_bn_relu" && !dropped_[i]) Fuse(i, true);
    std::vector<Instruction> out;
    for (size_t i = 0; i < instrs_.size(); ++i) {
      auto r = replacement_.find(i);
      if (r != replacement_.end()) {
        out.push_back(r->second);
      } else if (!dropped_[i]) {
        out.push_back(instrs_[i]);
      }
    }
    return Program(std::move(out), program_.GetInputs(), program_.name());
  }

 private:
  // what computes v, when it is an operator of this kind that is still there
  const Instruction* Source(const Variable& v, const char* op) const {
    auto it = defined_at_.find(v->id);
    return it == defined_at_.end() || instrs_[it->second]->op_type != op || dropped_[it->second] ? nullptr : &instrs_[it->second];
  }
  // the position of v's only reader, or -1
  int OnlyReader(const Variable& v) const {
    auto it = users_.find(v->id);
    return fetch_ids_.count(v->id) || it == users_.end() || it->second.size() != 1 ? -1 : static_cast<int>(it->second[0]);
  }
  // The chain of PaddleLayerNorm, walked from its result to its input; `chain_` collects its instructions.
  struct Norm {
    Variable x, gamma, beta;
    float epsilon;
  };
  const Instruction* Link(const Variable& v, const char* op, size_t inputs) {
    const Instruction* def = Source(v, op);
    if (!def || (*def)->inputs.size() != inputs) return nullptr;
    chain_.insert(defined_at_.at(v->id));
    return def;
  }
  // the operand of a broadcast of a vector along `axis`
  const Variable* Broadcast(const Variable& v, int axis) {
    const Instruction* def = Link(v, "broadcast_to", 1);
    return def && GetAttr<std::vector<int>>((*def)->attrs, "broadcast_axes", {}) == std::vector<int>{axis} ? &(*def)->inputs[0] : nullptr;
  }
  bool FillConstant(const Variable& v, float* value) {
    const Instruction* def = Link(v, "fill_constant", 0);
    if (def) *value = static_cast<float>(GetAttr<double>((*def)->attrs, "value", 0.0));
    return def != nullptr;
  }
  // v = sum over the rows of `of` / its columns
  bool IsMean(const Variable& v, const Variable& of) {
    const Instruction* div = Link(v, "divide", 2);
    float count            = 0.0f;
    if (!div || !FillConstant((*div)->inputs[1], &count) || count != static_cast<float>(of->shape[1])) return false;
    const Instruction* sum = Link((*div)->inputs[0], "reduce_sum", 1);
    return sum && (*sum)->inputs[0] == of && GetAttr<std::vector<int>>((*sum)->attrs, "dim", {}) == std::vector<int>{1};
  }
  // v = of * identity(of)
  bool IsSquare(const Variable& v, const Variable& of) {
    const Instruction* mul = Link(v, "elementwise_mul", 2);
    if (!mul || !((*mul)->inputs[0] == of)) return false;
    const Instruction* same = Link((*mul)->inputs[1], "identity", 1);
    return same && (*same)->inputs[0] == of;
  }
  bool MatchNorm(const Variable& y, Norm* norm) {
    chain_.clear();
    const Instruction* narrow = Link(y, "cast", 1);
    const Instruction* shaped = narrow ? Link((*narrow)->inputs[0], "reshape", 1) : nullptr;
    const Instruction* shift  = shaped ? Link((*shaped)->inputs[0], "elementwise_add", 2) : nullptr;
    const Instruction* scaled = shift ? Link((*shift)->inputs[0], "elementwise_mul", 2) : nullptr;
    const Instruction* div    = scaled ? Link((*scaled)->inputs[0], "divide", 2) : nullptr;
    if (!div) return false;
    const Variable *beta = Broadcast((*shift)->inputs[1], 1), *gamma = Broadcast((*scaled)->inputs[1], 1), *root = Broadcast((*div)->inputs[1], 0);
    const Instruction* centred = Link((*div)->inputs[0], "subtract", 2);
    const Variable* mean       = centred ? Broadcast((*centred)->inputs[1], 0) : nullptr;
    if (!beta || !gamma || !root || !mean) return false;
    const Variable& rows   = (*centred)->inputs[0];
    const Instruction* sq  = Link(*root, "sqrt", 1);
    const Instruction* eps = sq ? Link((*sq)->inputs[0], "elementwise_add", 2) : nullptr;
    const Instruction* var = eps ? Link((*eps)->inputs[0], "max", 2) : nullptr;
    float zero             = 1.0f;
    if (!var || !FillConstant((*eps)->inputs[1], &norm->epsilon) || !FillConstant((*var)->inputs[1], &zero) || zero != 0.0f) return false;
    const Instruction* diff = Link((*var)->inputs[0], "subtract", 2);
    if (!diff || rows->shape.size() != 2 || !IsMean(*mean, rows) || !IsSquare((*diff)->inputs[1], *mean)) return false;
    const Instruction* mean2 = Source((*diff)->inputs[0], "divide");
    const Instruction* sum2  = mean2 ? Source((*mean2)->inputs[0], "reduce_sum") : nullptr;
    if (!sum2 || !IsSquare((*sum2)->inputs[0], rows) || !IsMean((*diff)->inputs[0], (*sum2)->inputs[0])) return false;
    const Instruction* flat = Link(rows, "reshape", 1);
    const Instruction* wide = flat ? Link((*flat)->inputs[0], "cast", 1) : nullptr;
    // scale and bias before their conversion (which others may read too)
    const Instruction *g = Source(*gamma, "cast"), *b = Source(*beta, "cast");
    if (!wide || !g || !b) return false;
    norm->x = (*wide)->inputs[0], norm->gamma = (*g)->inputs[0], norm->beta = (*b)->inputs[0];
    const ShapeType& shape = rows->shape;
    if (!(norm->x->type == y->type) || !(norm->gamma->type == y->type) || !(norm->beta->type == y->type) || norm->x->shape != shape || y->shape != shape ||
        norm->gamma->shape != ShapeType{shape[1]} || norm->beta->shape != ShapeType{shape[1]})
      return false;
    // nothing else reads what is computed on the way
    for (size_t i : chain_) {
      for (auto& o : instrs_[i]->outputs) {
        if (o == y) continue;
        if (fetch_ids_.count(o->id)) return false;
        for (size_t u : users_[o->id])
          if (!chain_.count(u)) return false;
      }
    }
    return OnlyReader(y) >= 0;
  }

  // the slices that divide the columns of v, in order; empty if it is read in any other way
  std::vector<size_t> Columns(const Variable& v) const {
    auto it = users_.find(v->id);
    if (fetch_ids_.count(v->id) || it == users_.end() || it->second.size() < 2 || it->second.size() > 3) return {};
    std::vector<size_t> at = it->second;
    const int width        = v->shape[1] / static_cast<int>(at.size());
    if (width * static_cast<int>(at.size()) != v->shape[1]) return {};
    auto ints = [&](size_t i, const char* name) { return GetAttr<std::vector<int>>(instrs_[i]->attrs, name, {}); };
    for (size_t i : at) {
      const auto starts = ints(i, "starts"), ends = ints(i, "ends"), strides = ints(i, "strides");
      if (instrs_[i]->op_type != "slice" || dropped_[i] || ints(i, "axes") != std::vector<int>{1} || starts.size() != 1 || ends.size() != 1 ||
          !ints(i, "decrease_axis").empty() || !(strides.empty() || strides == std::vector<int>{1}) || starts[0] < 0 || starts[0] % width != 0 ||
          ends[0] != starts[0] + width || instrs_[i]->outputs[0]->shape != ShapeType{v->shape[0], width})
        return {};
    }
    std::sort(at.begin(), at.end(), [&](size_t a, size_t b) { return ints(a, "starts")[0] < ints(b, "starts")[0]; });
    for (size_t j = 0; j < at.size(); ++j)
      if (ints(at[j], "starts")[0] != static_cast<int>(j) * width) return {};
    return at;
  }

  // a transpose of v, through reshapes, that keeps the order of the axes longer than one
  void TransposesToReshapes(const Variable& v) {
    for (size_t i : users_[v->id]) {
      const auto& ins = instrs_[i];
      if (dropped_[i] || replacement_.count(i) || ins->outputs.size() != 1) continue;
      if (ins->op_type == "transpose") {
        const auto axes = GetAttr<std::vector<int>>(ins->attrs, "axis", {});
        int last        = -1;
        bool ordered    = axes.size() == v->shape.size();
        for (size_t a = 0; ordered && a < axes.size(); ++a) {
          if (axes[a] < 0 || axes[a] >= static_cast<int>(v->shape.size())) ordered = false;
          if (!ordered || v->shape[axes[a]] == 1) continue;
          ordered = axes[a] > last;
          last    = axes[a];
        }
        if (!ordered) continue;
        Instruction reshape("reshape");
        reshape->inputs  = ins->inputs;
        reshape->outputs = ins->outputs;
        reshape->attrs   = {{"shape", ins->outputs[0]->shape}};
        replacement_.emplace(i, reshape);
      } else if (ins->op_type == "reshape") {
        TransposesToReshapes(ins->outputs[0]);
      }
    }
  }

  // plain: also a layer with nothing to take along
  void Fuse(size_t at, bool plain) {
    const auto& conv = instrs_[at];
    if (conv->inputs.size() < 4 || conv->inputs.size() > 5 || conv->outputs.size() != 1 || GetAttr<bool>(conv->attrs, "relu", false) ||
        GetAttr<bool>(conv->attrs, "max_pool", false) || GetAttr<std::string>(conv->attrs, "data_format", "") != "NHWC")
      return;
    // a 1x1 filter may still look beside the one pixel (padding, and a stride that leaves one output)
    if (GetAttr<std::vector<int>>(conv->attrs, "stride", {1, 1}) != std::vector<int>{1, 1} ||
        GetAttr<std::vector<int>>(conv->attrs, "padding", {0, 0}) != std::vector<int>{0, 0} ||
        GetAttr<std::vector<int>>(conv->attrs, "dilation", {1, 1}) != std::vector<int>{1, 1} ||
        GetAttr<int>(conv->attrs, "groups", 1) != 1 || GetAttr<std::string>(conv->attrs, "input_layout", "NHWC") != "NHWC")
      return;
    // the layer's operands seen as 1x1 images
    auto matrix = [&](const Variable& image) -> const Variable* {
      const Instruction* def = Source(image, "reshape");
      const auto& s          = image->shape;
      if (!def || s.size() != 4 || s[1] != 1 || s[2] != 1 || (*def)->inputs[0]->shape != ShapeType{s[0], s[3]}) return nullptr;
      return &(*def)->inputs[0];
    };
    const Variable *w = matrix(conv->inputs[1]), *residual = conv->inputs.size() == 5 ? matrix(conv->inputs[4]) : nullptr;
    const Variable& x4 = conv->inputs[0];
    const int back     = OnlyReader(conv->outputs[0]);
    if (!matrix(x4) || !w || (conv->inputs.size() == 5 && !residual) || back < 0 || instrs_[back]->op_type != "reshape") return;
    Variable x = *matrix(x4), y = instrs_[back]->outputs[0];
    const int m = x->shape[0], k = x->shape[1], n = (*w)->shape[0];
    if (y->shape != ShapeType{m, n} || (*w)->shape[1] != k || (!x->type.is_float16() && !x->type.is_bfloat16())) return;
    if (m > 64 || k % 32 != 0 || static_cast<int64_t>(n) * k >= INT_MAX) return;

    Instruction call("hip_matmul_rows");
    call->inputs = {x, *w, conv->inputs[2], conv->inputs[3]};
    if (residual) call->inputs.push_back(*residual);
    std::vector<size_t> drop = {at, static_cast<size_t>(back)};
    size_t last              = static_cast<size_t>(back);

    Norm norm;
    const int reader = OnlyReader(y);
    cinn_hip_kernels::RowFusion fuse{k <= cinn_hip_kernels::kRowProductMaxNormK && OnlyReader(x4) >= 0 && MatchNorm(x, &norm),
                                     reader >= 0 && instrs_[reader]->op_type == "gelu" && !dropped_[reader]};
    std::vector<size_t> columns;
    if (!fuse.gelu && !residual) columns = Columns(y);
    cinn_hip_kernels::RowProduct product{};  // (a program's tensors are aligned)
    product.m = m, product.n = n, product.k = k;
    product.width   = columns.empty() ? n : n / static_cast<int>(columns.size());
    const bool ring = cinn_hip_kernels::RowRingTakes(product);
    fuse            = cinn_hip_kernels::ChooseRowFusion(m, n, k, ring, fuse);
    if (fuse.norm) {
      call->inputs[0] = norm.x;
      call->inputs.push_back(norm.gamma);
      call->inputs.push_back(norm.beta);
      drop.insert(drop.end(), chain_.begin(), chain_.end());
    }
    for (size_t j : {size_t(0), size_t(1), size_t(4)})  // the views as images
      if (j < conv->inputs.size() && OnlyReader(conv->inputs[j]) >= 0) drop.push_back(defined_at_.at(conv->inputs[j]->id));
    if (fuse.gelu) {
      y    = instrs_[reader]->outputs[0];
      last = static_cast<size_t>(reader);
      drop.push_back(last);
    }
    if (!fuse.norm && !fuse.gelu && !((plain || !columns.empty()) && cinn_hip_kernels::RowProductPays(m, n, k, ring, !columns.empty(), false))) return;
    if (columns.empty()) {
      call->outputs = {y};
    } else {
      // the call stands where the first of its results was
      last = *std::min_element(columns.begin(), columns.end());
      for (size_t c : columns) {
        call->outputs.push_back(instrs_[c]->outputs[0]);
        drop.push_back(c);
      }
    }
    call->attrs = {{"residual", residual != nullptr}, {"norm", fuse.norm}, {"gelu", fuse.gelu}, {"epsilon", fuse.norm ? norm.epsilon : 0.0f}};
    for (size_t d : drop) dropped_[d] = true;
    replacement_.emplace(last, call);
    for (auto& o : call->outputs) TransposesToReshapes(o);
  }

  const Program& program_;
  const std::set<std::string>& fetch_ids_;
  const std::vector<Instruction>& instrs_;
  std::vector<bool> dropped_;
  std::map<std::string, std::vector<size_t>> users_;
  std::map<std::string, size_t> defined_at_;
  std::set<size_t> chain_;
  std::map<size_t, Instruction> replacement_;
};

}  // namespace

Program FuseRowProducts(const Program& program, const std::set<std::string>& fetch_ids) {
  // the switch of the kernel that runs what is made here
  const char* skinny = getenv("FLAGS_cinn_hip_gemm_skinny");
  if (skinny && atoi(skinny) == 0) return program;
  return RowProductFuser(program, fetch_ids).Run();
}

}  // namespace frontend
}  // namespace cinn
