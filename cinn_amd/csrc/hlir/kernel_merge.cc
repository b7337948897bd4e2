#include "hlir/kernel_merge.h"

#include <algorithm>
#include <cstdlib>
#include <map>
#include <set>

#include "ir/ir_mutator.h"

namespace cinn {
namespace hlir {
namespace framework {

namespace {

using ir::Expr;

// a kernel whose body only knows its own blockIdx.x: one grid axis, every argument a buffer, no use of the grid size
bool Mergeable(const ir::LoweredFunc& f) {
  if (!f.is_device || !f.axis_info.valid) return false;
  if (f.axis_info.grid[1] != 1 || f.axis_info.grid[2] != 1) return false;
  for (auto& a : f.args)
    if (!a.is_buffer()) return false;
  for (const char* v : {"gridDim.x", "gridDim.y", "gridDim.z", "blockIdx.y", "blockIdx.z"})
    if (ir::UsesVar(f.body, v)) return false;
  return true;
}

// A block of bx x by threads whose body can run in a flat block of bx * by threads, with threadIdx.x and threadIdx.y
// recovered from the flat index: bx a power of two, no third axis, no use of the block's extents (the device library's
// wave and block reductions work on the linear thread index; the column reduction walks blockDim.y and is excluded
// by the group kinds that get here).
bool Flattenable(const Group& g, const ir::LoweredFunc& f) {
  if (g.kind != GroupKind::kElementwise && g.kind != GroupKind::kRowReduce) return false;
  const int bx = f.axis_info.block[0];
  if (f.axis_info.block[2] != 1 || bx <= 0 || (bx & (bx - 1)) != 0) return false;
  for (const char* v : {"blockDim.x", "blockDim.y", "blockDim.z", "threadIdx.z"})
    if (ir::UsesVar(f.body, v)) return false;
  return true;
}

int Threads(const ir::LoweredFunc& f) { return f.axis_info.block[0] * f.axis_info.block[1] * f.axis_info.block[2]; }

// what decides which groups share a launch
struct MergeTraits {
  const Group* group;
  bool mergeable{false}, flattenable{false};
  int block[3]{0, 0, 0}, threads{0};
  int64_t grid{0};
};

std::vector<MergeTraits> TraitsOf(const std::vector<std::unique_ptr<Group>>& groups, const std::vector<ir::LoweredFuncRef>& funcs,
                                  const std::vector<bool>& barrier, const KernelMergeOptions& options) {
  std::vector<MergeTraits> traits;
  for (size_t i = 0; i < groups.size(); ++i) {
    MergeTraits t;
    t.group     = groups[i].get();
    t.mergeable = options.enabled && !barrier[i] && Mergeable(*funcs[i]);
    if (t.mergeable) {
      t.flattenable = Flattenable(*groups[i], *funcs[i]);
      for (int d = 0; d < 3; ++d) t.block[d] = funcs[i]->axis_info.block[d];
      t.threads = Threads(*funcs[i]);
      t.grid    = funcs[i]->axis_info.grid[0];
    }
    traits.push_back(t);
  }
  return traits;
}

bool SameBlock(const MergeTraits& a, const MergeTraits& b) { return std::equal(a.block, a.block + 3, b.block); }

bool Reads(const Group& g, const Group& writer) {
  for (auto* in : g.inputs)
    for (auto* out : writer.outputs)
      if (in == out) return true;
  return false;
}

// the program input that a group sees in `v`: `v` itself, or what it is a reshape (a view) of; null for a computed value
const NodeData* ProgramInput(const NodeData* v) {
  while (v->producer && v->producer->op_type() == "reshape") v = v->producer->inputs[0];
  return v->producer ? nullptr : v;
}

// a value that the program returns, itself or through reshapes
bool IsResult(const NodeData* v) {
  if (v->is_fetch || v->consumers.empty()) return true;
  for (auto* n : v->consumers)
    if (n->op_type() == "reshape" && IsResult(n->outputs[0])) return true;
  return false;
}

// `g` reads a program input that `reader` reads and writes a result of its type and size: a caller may have bound that
// result to the input's memory, an update in place, and what `reader` sees depends on which of the two comes first.
bool MayUpdate(const Group& g, const Group& reader) {
  for (auto* read : reader.inputs) {
    const NodeData* input = ProgramInput(read);
    if (!input || std::none_of(g.inputs.begin(), g.inputs.end(), [&](const NodeData* in) { return ProgramInput(in) == input; })) continue;
    for (auto* out : g.outputs)
      if (IsResult(out) && out->dtype == input->dtype && out->numel() == input->numel()) return true;
  }
  return false;
}

// Whether two groups that are not ordered by a value still keep their order, so that no launch runs their blocks side by side:
// one may update what the other reads, element by element; or in any way, unless the program itself has the two next to
// each other (a softmax and a maximum of one input have always shared a launch there).
bool KeepOrder(const Group& a, const Group& b) {
  const bool updates = MayUpdate(a, b), updated = MayUpdate(b, a);
  if (!updates && !updated) return false;
  return (updates && a.kind == GroupKind::kElementwise) || (updated && b.kind == GroupKind::kElementwise) || a.program_run != b.program_run;
}

// One behind the last group of the run that begins at t[i]: the longest run of consecutive kernels none of which reads what an
// earlier one of the run writes, or keeps its order for another reason; the run is
// consecutive in execution order, so a dependence through other groups would pass through a member as well.
size_t RunEnd(const std::vector<MergeTraits>& t, size_t i, const KernelMergeOptions& options) {
  if (!t[i].mergeable) return i + 1;
  int64_t blocks = t[i].grid;
  size_t end     = i + 1;
  // A run keeps one block shape, or - once a member of another shape joins - every member must be able to run in a
  // flat block of the same number of threads (a member that cannot, e.g. a column reduction, shares launches only
  // with kernels of its own shape).
  bool run_flat        = false;
  bool all_flattenable = t[i].flattenable;
  while (end < t.size() && static_cast<int>(end - i) < options.max_members) {
    if (!t[end].mergeable || t[end].group->pre_run != t[i].group->pre_run) break;
    const bool same = SameBlock(t[i], t[end]);
    if ((run_flat || !same) && (!all_flattenable || !t[end].flattenable || t[i].threads != t[end].threads)) break;
    bool depends = false;
    for (size_t k = i; k < end; ++k)
      depends |= Reads(*t[end].group, *t[k].group) || KeepOrder(*t[end].group, *t[k].group);
    if (depends) break;
    if (blocks + t[end].grid > 0x7fffffff) break;
    blocks += t[end].grid;
    run_flat        = run_flat || !same;
    all_flattenable = all_flattenable && t[end].flattenable;
    ++end;
  }
  return end;
}

// launches of the groups from `first` to before `last`
int Launches(const std::vector<MergeTraits>& t, size_t first, size_t last, const KernelMergeOptions& options) {
  int n = 0;
  for (size_t i = first; i < last; i = RunEnd(t, i, options)) ++n;
  return n;
}

// whether two groups that are not ordered by a value may change places
bool MayPass(const Group& a, const Group& b) {
  return !Reads(a, b) && !Reads(b, a) && !MayUpdate(a, b) && !MayUpdate(b, a);
}

LaunchUnit UnitOf(const Group& g) {
  LaunchUnit u;
  u.func_name = g.func_name;
  u.inputs    = g.inputs;
  u.outputs   = g.outputs;
  u.pre_run   = g.pre_run;
  u.members   = {&g};
  return u;
}

}  // namespace

std::vector<size_t> OrderForMerging(const std::vector<std::unique_ptr<Group>>& groups, const std::vector<ir::LoweredFuncRef>& funcs,
                                    const std::vector<bool>& barrier, const KernelMergeOptions& options) {
  CINN_CHECK_EQ(groups.size(), funcs.size());
  std::vector<size_t> order(groups.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = i;
  std::vector<MergeTraits> t = TraitsOf(groups, funcs, barrier, options);
  for (auto& g : groups) g->program_run = -1;
  for (size_t i = 0, run = 0; i < t.size(); ++run)
    for (const size_t end = RunEnd(t, i, options); i < end; ++i) groups[i]->program_run = static_cast<int>(run);
  auto small = [&](const MergeTraits& m) {
    int64_t bytes = 0;
    for (auto* list : {&m.group->inputs, &m.group->outputs})
      for (auto* v : *list) bytes += v->numel() * v->dtype.bytes();
    return m.mergeable && !m.group->pre_run && bytes <= options.max_moved_bytes;
  };
  auto move = [](auto* list, size_t from, size_t to) {
    if (from < to) std::rotate(list->begin() + from, list->begin() + from + 1, list->begin() + to + 1);
    if (to < from) std::rotate(list->begin() + to, list->begin() + from, list->begin() + from + 1);
  };
  // how far a group looks, and how many places it tries in either direction: a program of thousands of groups is ordered in
  // a time that grows with their number
  constexpr size_t kReach = 64;
  constexpr int kPlaces   = 8;
  const size_t around     = options.max_members;
  for (size_t group = 0; group < order.size(); ++group) {
    size_t at = std::find(order.begin(), order.end(), group) - order.begin();
    if (!small(t[at])) continue;
    // the nearest place, later or earlier, that saves a launch: next to a kernel, past groups that it may change places with
    bool moved = false;
    int places = 0;
    auto attempt = [&](size_t to) {
      const size_t low = std::min(at, to), first = low > around ? low - around : 0, last = std::min(t.size(), std::max(at, to) + 1 + around);
      const int before = Launches(t, first, last, options);
      move(&t, at, to);
      moved = Launches(t, first, last, options) < before;
      if (moved) {
        move(&order, at, to);
      } else {
        move(&t, to, at);
      }
      ++places;
    };
    const size_t end = std::min(t.size(), at + 1 + kReach), begin = at > kReach ? at - kReach : 0;
    for (size_t to = at + 1; to < end && !moved && places < kPlaces && MayPass(*t[at].group, *t[to].group); ++to)
      if (to + 1 < t.size() && t[to + 1].mergeable) attempt(to);
    places = 0;
    for (size_t to = at; to-- > begin && !moved && places < kPlaces && MayPass(*t[at].group, *t[to].group);)
      if (to > 0 && t[to - 1].mergeable) attempt(to);
  }
  return order;
}

std::vector<LaunchUnit> MergeIndependentKernels(const std::vector<std::unique_ptr<Group>>& groups,
                                                const std::vector<ir::LoweredFuncRef>& funcs, const std::vector<bool>& barrier,
                                                const KernelMergeOptions& options, std::vector<ir::LoweredFuncRef>* funcs_out) {
  CINN_CHECK_EQ(groups.size(), funcs.size());
  const std::vector<MergeTraits> traits = TraitsOf(groups, funcs, barrier, options);
  std::vector<LaunchUnit> units;
  size_t i = 0;
  while (i < groups.size()) {
    const Group& first = *groups[i];
    const size_t end = RunEnd(traits, i, options);
    if (end - i < 2) {  // not mergeable, or alone
      units.push_back(UnitOf(first));
      funcs_out->push_back(funcs[i]);
      ++i;
      continue;
    }
    // one kernel: parameters are the members' inputs (each value once) followed by their outputs
    LaunchUnit unit;
    unit.pre_run = first.pre_run;
    auto merged  = std::make_shared<ir::LoweredFunc>();
    merged->is_device = true;
    merged->axis_info = funcs[i]->axis_info;
    int64_t blocks = 0;
    for (size_t k = i; k < end; ++k) blocks += traits[k].grid;
    merged->axis_info.grid[0] = static_cast<int>(blocks);
    // members of different block shapes: the launch is a flat block and every member recovers its own threadIdx.x / y
    bool flat = false;
    for (size_t k = i + 1; k < end; ++k) flat = flat || !SameBlock(traits[i], traits[k]);
    if (flat) {
      merged->axis_info.block[0] = funcs[i]->axis_info.block[0] * funcs[i]->axis_info.block[1];
      merged->axis_info.block[1] = 1;
    }
    merged->name = first.func_name + "_and_" + std::to_string(end - i - 1) + "_more";
    std::map<std::string, ir::Argument> arg_of;  // by buffer name: the first member's buffer object is declared
    for (size_t k = i; k < end; ++k) {
      unit.members.push_back(groups[k].get());
      for (auto& a : funcs[k]->args) arg_of.emplace(a.buffer->name, a);
    }
    std::set<const NodeData*> seen;
    std::vector<ir::Argument> ins, outs;
    for (size_t k = i; k < end; ++k) {
      const Group& g = *groups[k];
      CINN_CHECK_EQ(funcs[k]->args.size(), g.inputs.size() + g.outputs.size());
      for (size_t a = 0; a < g.inputs.size(); ++a) {
        if (!seen.insert(g.inputs[a]).second) continue;
        unit.inputs.push_back(g.inputs[a]);
        ins.push_back(arg_of.at(funcs[k]->args[a].buffer->name));
        ins.back().io = ir::Argument::IO::kInput;
      }
      for (size_t a = 0; a < g.outputs.size(); ++a) {
        unit.outputs.push_back(g.outputs[a]);
        outs.push_back(funcs[k]->args[g.inputs.size() + a]);
        outs.back().io = ir::Argument::IO::kOutput;
      }
    }
    merged->args = ins;
    merged->args.insert(merged->args.end(), outs.begin(), outs.end());
    // bodies: block b of the launch is block b - start of the member whose range holds it.  Blocks are dispatched in
    // index order: the member with the most blocks comes first, so that the launch ends on short members
    // (measured on six members of 2048 - 4096 blocks: within 0.5 % of program order and of the reverse;
    // FLAGS_cinn_hip_merge_order = 0: program order, 2: fewest blocks first).
    std::vector<size_t> order;
    for (size_t k = i; k < end; ++k) order.push_back(k);
    static const int order_flag = [] {
      const char* v = getenv("FLAGS_cinn_hip_merge_order");
      return v && *v ? atoi(v) : 1;
    }();
    if (order_flag == 1 || order_flag == 2)
      std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) {
        return order_flag == 1 ? funcs[a]->axis_info.grid[0] > funcs[b]->axis_info.grid[0]
                               : funcs[a]->axis_info.grid[0] < funcs[b]->axis_info.grid[0];
      });
    Expr block_x = ir::MakeVar("blockIdx.x", common::Int(32));
    Expr chain;
    int64_t start = blocks;
    for (size_t pos = order.size(); pos-- > 0;) {
      const size_t k = order[pos];
      start -= funcs[k]->axis_info.grid[0];
      // temporaries are declared once at the top of the kernel: keep the members' names apart
      for (auto& buf : funcs[k]->temp_bufs) {
        buf->name = "m" + std::to_string(k - i) + "_" + buf->name;
        merged->temp_bufs.push_back(buf);
      }
      Expr body = start == 0 ? funcs[k]->body : ir::Substitute(funcs[k]->body, "blockIdx.x", block_x - Expr(static_cast<int>(start)));
      if (flat && funcs[k]->axis_info.block[1] > 1) {
        const int bx = funcs[k]->axis_info.block[0];
        int shift    = 0;
        while ((1 << shift) < bx) ++shift;
        const std::string tag = "m" + std::to_string(k - i);
        Expr tx = ir::MakeVar(tag + "_tx", common::Int(32)), ty = ir::MakeVar(tag + "_ty", common::Int(32));
        Expr tid = ir::MakeVar("threadIdx.x", common::Int(32));
        body = ir::Substitute(ir::Substitute(body, "threadIdx.x", tx), "threadIdx.y", ty);
        body = ir::MakeBlock({ir::MakeLet(tx, tid % Expr(bx)), ir::MakeLet(ty, tid / Expr(bx)), body});
      }
      if (!chain.defined()) {
        chain = ir::MakeBlock({body});  // the last member takes every remaining block
      } else {
        chain = ir::MakeIf(block_x < Expr(static_cast<int>(start + funcs[k]->axis_info.grid[0])), ir::MakeBlock({body}), chain);
      }
    }
    merged->body   = chain;
    unit.func_name = merged->name;
    funcs_out->push_back(merged);
    units.push_back(unit);
    i = end;
  }
  return units;
}

}  // namespace framework
}  // namespace hlir
}  // namespace cinn
