#include "hip_planner.h"

// Operations along the last axis that the op library composes from several, planned as one launch each.

namespace pmlc::target::hip {

namespace {
int64_t rowsOf(const TensorShape& s) {
  return s.sizes.back() ? static_cast<int64_t>(s.elements()) / s.sizes.back() : 0;
}
}  // namespace

// every use of v lies in `users`, none is an output of the program, none is planned already
bool Planner::usedOnlyBy(const ValuePtr& v, const std::set<size_t>& users) {
  if (outputs_.count(v.get())) return false;
  const auto it = users_.find(v.get());
  if (it == users_.end()) return false;
  for (size_t u : it->second)
    if (!users.count(u) || consumed_.count(u)) return false;
  return true;
}

// The op library's argmax (plaidml/op/lib/ops.cc:505-521) over the last axis: M = max of the row, P = max over the row of
// cond(x, M, index) -- the last position that holds the maximum -- and a cast to an unsigned type of the same width, which
// changes no bit.  `i` is the first contraction.
bool Planner::tryArgmax(size_t i) {
  Op& mx = prog_->ops[i];
  if (mx.kind != Op::Contraction || mx.agg != AggKind::max || mx.combo != ComboKind::none || mx.operands.size() != 1 || mx.init || !mx.constraints.empty()) return false;
  const ValuePtr X = mx.operands[0];
  const DataType dt = X->shape.elementType;
  if ((dt != DataType::f32 && dt != DataType::bf16) || mx.result->shape.elementType != dt || X->kind == Value::Literal) return false;
  const size_t r = X->shape.getRank();
  if (r < 1 || mx.accesses.size() != 2 || mx.accesses[1].size() != r || mx.idxNames.size() != r) return false;
  const auto uit = users_.find(mx.result.get());
  if (uit == users_.end() || uit->second.empty()) return false;
  const size_t pi = uit->second.front();
  if (!usedOnlyBy(mx.result, {pi})) return false;
  Op& pos = prog_->ops[pi];
  if (pos.kind != Op::Contraction || pos.agg != AggKind::max || pos.combo != ComboKind::cond || pos.operands.size() != 3 || pos.init ||
      !pos.constraints.empty() || pos.operands[0] != X || pos.operands[1] != mx.result || pos.accesses.size() != 4 || pos.idxNames.size() != r)
    return false;
  if (pos.result->shape.elementType != DataType::si32 || pos.result->shape.sizes != mx.result->shape.sizes) return false;
  const auto ix = producer_.find(pos.operands[2].get());
  if (ix == producer_.end() || prog_->ops[ix->second].kind != Op::Index) return false;
  const Op& index = prog_->ops[ix->second];
  if (index.axis != 0 || pos.operands[2]->shape.sizes != std::vector<int64_t>{X->shape.sizes[r - 1]}) return false;
  if (!pos.boundsComputed) tile::computeBounds(&pos);
  // both walk the whole of X with an index per dimension; the result keeps all of them but the last, in order
  for (const Op* op : {static_cast<const Op*>(&mx), static_cast<const Op*>(&pos)}) {
    if (emptyBox(*op)) return false;
    std::vector<int> idx(r);
    for (size_t d = 0; d < r; ++d) {
      idx[d] = op->accesses[1][d].plainIndex();
      if (idx[d] < 0 || op->lower[idx[d]] != 0 || op->upper[idx[d]] != X->shape.sizes[d] - 1) return false;
      for (size_t e = 0; e < d; ++e)
        if (idx[e] == idx[d]) return false;
    }
    // the result's access: the leading indices, with or without a constant 0 in the last axis' place
    auto leading = [&](const std::vector<Affine>& a) {
      if (a.size() != r - 1 && a.size() != r) return false;
      for (size_t d = 0; d + 1 < r; ++d)
        if (a[d].plainIndex() != idx[d]) return false;
      return a.size() == r - 1 || (a[r - 1].isConstant() && a[r - 1].c0 == 0);
    };
    if (!leading(op->accesses[0])) return false;
    if (op == &pos && (!leading(op->accesses[2]) || op->accesses[3].size() != 1 || op->accesses[3][0].plainIndex() != idx[r - 1])) return false;
  }
  if (static_cast<int64_t>(mx.result->shape.elements()) != rowsOf(X->shape)) return false;
  ValuePtr out = pos.result;
  std::set<size_t> taken = {pi};
  const auto pu = users_.find(pos.result.get());
  if (!outputs_.count(pos.result.get()) && pu != users_.end() && pu->second.size() == 1 && !consumed_.count(pu->second[0])) {
    const Op& c = prog_->ops[pu->second[0]];
    if (c.kind == Op::Cast && (c.result->shape.elementType == DataType::ui32 || c.result->shape.elementType == DataType::si32)) {
      out = c.result;
      taken.insert(pu->second[0]);
    }
  }
  Step s;
  s.kind = Step::Argmax;
  s.sm.dtype = hipType(dt);
  s.sm.cols = X->shape.sizes[r - 1];
  s.sm.rows = rowsOf(X->shape);
  s.a = bufferFor(X);
  s.c = bufferFor(out);
  consumed_.insert(taken.begin(), taken.end());
  s.bytes = static_cast<double>(X->shape.getByteSize() + out->shape.getByteSize());
  s.text = "argmax " + std::string(util::mnemonic(dt)) + " over the last axis of " + X->shape.str() + " -> " + out->shape.str();
  plan_->steps.push_back(s);
  return true;
}

// Whether `taken` is X's elements in the order `order` names along the last axis, as the op library's sort composes it
// (plaidml/op/lib/ops.cc: gather of X at coordinates [.., rank] that are the sum of one assignment per dimension: the
// dimension's own index, or `order` in the last one).  Collects the operations in between.
bool Planner::isTakenInOrder(const ValuePtr& taken, const ValuePtr& X, const ValuePtr& order, std::set<size_t>* between) {
  auto made_by = [&](const ValuePtr& v) -> size_t {
    const auto it = producer_.find(v.get());
    return it == producer_.end() ? std::string::npos : it->second;
  };
  const size_t gi = made_by(taken);
  if (gi == std::string::npos) return false;
  const Op& g = prog_->ops[gi];
  const size_t r = X->shape.getRank();
  if (g.kind != Op::Special || g.fn != "gather" || g.operands.size() != 2 || g.operands[0] != X || g.params.size() != 7 ||
      g.params[4] != PML_HIP_GATHER_ND || g.params[5] != 0 || g.result->shape.sizes != X->shape.sizes)
    return false;
  between->insert(gi);
  std::vector<bool> seen(r, false);
  std::vector<ValuePtr> todo = {g.operands[1]};
  while (!todo.empty()) {
    const ValuePtr v = todo.back();
    todo.pop_back();
    const size_t vi = made_by(v);
    if (vi == std::string::npos) return false;
    Op& op = prog_->ops[vi];
    between->insert(vi);
    if (op.kind == Op::Eltwise && op.fn == "add" && op.operands.size() == 2) {
      for (const ValuePtr& o : op.operands) {
        if (o->kind == Value::Literal || o->shape.sizes != v->shape.sizes || o->shape.elementType != DataType::si32) return false;
        todo.push_back(o);
      }
      continue;
    }
    // C[x0, .., xr-1, xr + d] = S[x0, .., xr-1, xr] with S one value per element: column d of the coordinates
    if (op.kind != Op::Contraction || op.agg != AggKind::assign || op.combo != ComboKind::none || op.operands.size() != 1 || op.init ||
        !op.constraints.empty() || op.accesses.size() != 2 || op.accesses[0].size() != r + 1 || op.accesses[1].size() != r + 1)
      return false;
    const TensorShape& src = op.operands[0]->shape;
    if (src.getRank() != r + 1 || src.sizes[r] != 1 || op.result->shape.sizes[r] != static_cast<int64_t>(r) || src.elementType != DataType::si32) return false;
    std::set<int> idx;
    for (size_t d = 0; d < r; ++d) {
      const int v0 = op.accesses[0][d].plainIndex();
      if (v0 < 0 || op.accesses[1][d].plainIndex() != v0 || !idx.insert(v0).second || src.sizes[d] != X->shape.sizes[d]) return false;
    }
    const int last = op.accesses[1][r].plainIndex();
    Affine col = op.accesses[0][r];
    if (last < 0 || idx.count(last) || col.den != 1) return false;
    const int64_t d = col.c0;
    col.c0 = 0;
    if (col.plainIndex() != last || d < 0 || d >= static_cast<int64_t>(r) || seen[static_cast<size_t>(d)]) return false;
    seen[static_cast<size_t>(d)] = true;
    const size_t ri = made_by(op.operands[0]);
    if (ri == std::string::npos || prog_->ops[ri].kind != Op::Reshape) return false;
    between->insert(ri);
    const ValuePtr& from = prog_->ops[ri].operands[0];
    if (from->shape.sizes != X->shape.sizes) return false;
    if (d + 1 == static_cast<int64_t>(r)) {
      if (from != order) return false;
    } else {
      const size_t xi = made_by(from);
      if (xi == std::string::npos || prog_->ops[xi].kind != Op::Index || prog_->ops[xi].axis != d) return false;
      between->insert(xi);
    }
  }
  for (size_t d = 0; d < r; ++d)
    if (!seen[d]) return false;
  return true;
}

// The first k of a sort along the last axis (plaidml/op/lib/ops.cc:2420-2467): an argsort whose result is used by a gather
// of its first k entries, and / or by the sort composition whose result's first k entries are gathered.  `i` is the argsort.
bool Planner::tryTopk(size_t i) {
  const Op& as = prog_->ops[i];
  const ValuePtr X = as.operands[0], order = as.result;
  const size_t r = X->shape.getRank();
  const DataType dt = X->shape.elementType;
  if (r < 1 || util::byteSize(dt) > 4 || X->kind == Value::Literal || outputs_.count(order.get())) return false;
  int64_t axis = static_cast<int64_t>(as.params.at(0));
  if (axis < 0) axis += static_cast<int64_t>(r);
  if (axis != static_cast<int64_t>(r) - 1 || X->shape.sizes[r - 1] > PML_HIP_MAX_SORT_LINE || X->shape.elements() == 0) return false;
  // a gather along the last axis by index({k}, 0): the first k entries
  auto firstEntries = [&](size_t u, const ValuePtr& of, int64_t* k) {
    const Op& g = prog_->ops[u];
    if (g.kind != Op::Special || g.fn != "gather" || g.operands.size() != 2 || g.operands[0] != of || g.params.size() != 7) return false;
    int64_t ax = static_cast<int64_t>(g.params[0]);
    if (ax < 0) ax += static_cast<int64_t>(r);
    if (ax != axis || g.params[4] != PML_HIP_GATHER_NORMAL) return false;
    const auto it = producer_.find(g.operands[1].get());
    if (it == producer_.end() || prog_->ops[it->second].kind != Op::Index || g.operands[1]->shape.getRank() != 1) return false;
    *k = g.operands[1]->shape.sizes[0];
    return *k > 0 && *k <= X->shape.sizes[r - 1] && g.result->shape.getRank() == r && g.result->shape.sizes[r - 1] == *k;
  };
  int64_t k = 0;
  size_t pos_gather = std::string::npos, val_gather = std::string::npos;
  std::set<size_t> between, order_users;
  const auto uit = users_.find(order.get());
  if (uit == users_.end()) return false;
  for (size_t u : uit->second) {
    if (consumed_.count(u)) return false;
    order_users.insert(u);
  }
  for (size_t u : order_users) {
    int64_t kk = 0;
    if (pos_gather == std::string::npos && firstEntries(u, order, &kk)) {
      pos_gather = u;
      k = kk;
    }
  }
  order_users.erase(pos_gather);
  if (order_users.size() > 1) return false;
  if (order_users.size() == 1) {
    // the reshape at the start of the sort composition: find the gather of X that ends it
    const auto xu = users_.find(X.get());
    for (size_t u : xu->second) {
      std::set<size_t> ops;
      const ValuePtr sorted = prog_->ops[u].result;
      if (consumed_.count(u) || !isTakenInOrder(sorted, X, order, &ops) || !ops.count(*order_users.begin())) continue;
      const auto su = users_.find(sorted.get());
      int64_t kk = 0;
      if (outputs_.count(sorted.get()) || su == users_.end() || su->second.size() != 1 || !firstEntries(su->second[0], sorted, &kk)) return false;
      if (pos_gather != std::string::npos && kk != k) return false;
      k = kk;
      val_gather = su->second[0];
      between = ops;
      break;
    }
    if (val_gather == std::string::npos) return false;
    // nothing in between may serve anything else (indices may: they are made again where needed)
    std::set<size_t> inside = between;
    inside.insert(val_gather);
    // (some of it comes before the argsort and has been planned: with no user left those launches are dropped)
    for (size_t b : between) {
      if (prog_->ops[b].kind == Op::Index) continue;
      if (outputs_.count(prog_->ops[b].result.get())) return false;
      for (size_t u : users_[prog_->ops[b].result.get()])
        if (!inside.count(u)) return false;
    }
  }
  if (k <= 0 || k > 128) return false;  // (a wavefront picks them one after the other: beyond that the sort is cheaper)
  Step s;
  s.kind = Step::TopK;
  s.sm.dtype = hipType(dt);
  s.sm.cols = X->shape.sizes[r - 1];
  s.sm.rows = rowsOf(X->shape);
  s.topk = static_cast<int>(k);
  s.topk_descending = static_cast<int64_t>(as.params.at(1)) != 0;
  s.a = bufferFor(X);
  s.c = val_gather == std::string::npos ? -1 : bufferFor(prog_->ops[val_gather].result);
  s.out2 = pos_gather == std::string::npos ? -1 : bufferFor(prog_->ops[pos_gather].result);
  for (size_t u : {pos_gather, val_gather})
    if (u != std::string::npos) consumed_.insert(u);
  for (size_t b : between)
    if (prog_->ops[b].kind != Op::Index) consumed_.insert(b);
  consumed_.insert(i);
  s.bytes = static_cast<double>(X->shape.getByteSize()) + static_cast<double>(s.sm.rows * k) * (4 + util::byteSize(dt));
  s.text = "top " + std::to_string(k) + (s.topk_descending ? " desc" : " asc") + " of the last axis of " + X->shape.str() + (s.c >= 0 ? " values" : "") +
           (s.out2 >= 0 ? " positions" : "");
  plan_->steps.push_back(s);
  return true;
}

// A region of element-wise operations and reductions along the last axis that share one matrix shape [.., C], starting with
// the reduction `i`: one launch of a row program in place of a launch per reduction and per element-wise chain (the op
// library's mvn and normalisations: ten launches).  Operations join in program order while every operand is a value of the
// region or existed before it; the values nothing inside reads are its results.
bool Planner::tryRowProgram(size_t i) {
  const Op& first = prog_->ops[i];
  // the aggregation of a reduction along the last axis, or -1
  auto rowReduction = [&](const Op& op) {
    if (op.operands.size() != 1 || op.operands[0]->kind == Value::Literal) return -1;
    for (AggKind a : {AggKind::add, AggKind::mul, AggKind::max, AggKind::min})
      if (reducesLastAxis(op, a)) return hipAgg(a);
    return -1;
  };
  if (rowReduction(first) < 0) return false;
  const TensorShape shape = first.operands[0]->shape;
  const DataType dt = shape.elementType;
  if ((dt != DataType::f32 && dt != DataType::bf16) || shape.getRank() < 2 || shape.elements() == 0) return false;
  const size_t r = shape.getRank();
  TensorShape row_shape = shape;
  row_shape.sizes[r - 1] = 1;
  const bool one_col = shape.sizes[r - 1] == 1;
  if (one_col) return false;
  auto isFull = [&](const ValuePtr& v) { return v->kind != Value::Literal && v->shape.sizes == shape.sizes && v->shape.elementType == dt; };
  auto isRow = [&](const ValuePtr& v) { return v->kind != Value::Literal && v->shape.sizes == row_shape.sizes && v->shape.elementType == dt; };

  struct Node {
    size_t op;
    bool row;
    int opcode;  // EPI opcode, or aggregation of a reduction
    bool reduce;
    ValuePtr a, b;  // b null: none, or the immediate
    bool imm;
    double imm_value;
  };
  std::vector<Node> nodes;
  std::map<const Value*, size_t> made;        // region value -> node
  std::map<const Value*, const Value*> same;  // a value computed twice -> its first computation
  auto canon = [&](const ValuePtr& v) -> const Value* {
    const auto it = same.find(v.get());
    return it == same.end() ? v.get() : it->second;
  };
  static const std::set<int> usable = {PML_HIP_EPI_ADD, PML_HIP_EPI_SUB, PML_HIP_EPI_RSUB, PML_HIP_EPI_MUL, PML_HIP_EPI_DIV,
                                       PML_HIP_EPI_RDIV, PML_HIP_EPI_MAX, PML_HIP_EPI_MIN, PML_HIP_EPI_RELU, PML_HIP_EPI_NEG,
                                       PML_HIP_EPI_EXP, PML_HIP_EPI_LOG, PML_HIP_EPI_SQRT, PML_HIP_EPI_TANH, PML_HIP_EPI_MAX_GT};
  // operand classes a node may read
  auto readable = [&](const ValuePtr& v, bool row) {
    if (made.count(canon(v))) return !row || prog_->ops[nodes[made[canon(v)]].op].result->shape.sizes == row_shape.sizes;
    if (v->shape.elementType != dt) return false;
    if (v->kind == Value::Temp) {
      const auto it = producer_.find(v.get());
      if (it == producer_.end() || it->second >= i || !bufferOf_.count(v.get())) return false;
    }
    if (v->shape.elements() == 1 || isRow(v)) return true;
    if (row) return false;
    if (isFull(v)) return true;
    // one value per column
    if (v->shape.getRank() < 1 || v->shape.getRank() > r || v->shape.sizes.back() != shape.sizes[r - 1]) return false;
    for (size_t d = 0; d + 1 < v->shape.getRank(); ++d)
      if (v->shape.sizes[d] != 1) return false;
    return true;
  };
  size_t reductions = 0;
  for (size_t j = i; j < prog_->ops.size() && nodes.size() < PML_HIP_ROWS_STEPS; ++j) {
    if (j != i && consumed_.count(j)) continue;
    Op& op = prog_->ops[j];
    Node n{j, false, 0, false, nullptr, nullptr, false, 0};
    if (op.kind == Op::Contraction) {
      if (op.operands.size() != 1 || op.operands[0]->kind == Value::Literal || op.operands[0]->shape.sizes != shape.sizes) continue;
      if (!op.boundsComputed) tile::computeBounds(&op);
      const int agg = rowReduction(op);
      if (agg < 0 || op.operands[0]->shape.elementType != dt || !readable(op.operands[0], false)) continue;
      n.row = n.reduce = true;
      n.opcode = agg;
      n.a = op.operands[0];
      double f = 0;
      int64_t unused = 0;
      tile::aggregationIdentity(op.agg, dt, &f, &unused);
      n.imm_value = f;
    } else if (op.kind == Op::Eltwise && op.result->shape.elementType == dt) {
      n.row = op.result->shape.sizes == row_shape.sizes;
      if (!n.row && op.result->shape.sizes != shape.sizes) continue;
      if (op.operands.size() == 1) {
        n.opcode = unaryOpcode(op.fn);
        n.a = op.operands[0];
      } else if (op.operands.size() == 2) {
        const bool lead = op.operands[0]->kind != Value::Literal;
        n.opcode = binaryOpcode(op.fn, lead);
        n.a = op.operands[lead ? 0 : 1];
        const ValuePtr& o = op.operands[lead ? 1 : 0];
        if (o->kind == Value::Literal) {
          n.imm = true;
          n.imm_value = o->literalAsDouble();
        } else {
          n.b = o;
        }
      }
      if (!n.a || n.a->kind == Value::Literal || !usable.count(n.opcode) || !readable(n.a, n.row) || (n.b && !readable(n.b, n.row))) continue;
      // at least one operand from the region: other element-wise operations keep their own launches
      if (!made.count(canon(n.a)) && !(n.b && made.count(canon(n.b)))) continue;
    } else {
      continue;
    }
    // the same operation on the same operands: one value
    bool twin = false;
    for (const Node& m : nodes)
      if (m.reduce == n.reduce && m.opcode == n.opcode && canon(m.a) == canon(n.a) && (m.b ? canon(m.b) : nullptr) == (n.b ? canon(n.b) : nullptr) &&
          m.imm == n.imm && m.imm_value == n.imm_value && m.row == n.row && !outputs_.count(op.result.get())) {
        same[op.result.get()] = prog_->ops[m.op].result.get();
        twin = true;
        break;
      }
    reductions += n.reduce;
    if (!twin) made[op.result.get()] = nodes.size();
    nodes.push_back(n);
    if (twin) nodes.back().reduce = n.reduce, nodes.back().opcode = -1;  // (kept to be consumed; emits nothing)
  }
  size_t work = 0;
  for (const Node& n : nodes) work += n.opcode != -1;
  if (work < 3) return false;

  std::set<size_t> members;
  for (const Node& n : nodes) members.insert(n.op);
  // values that leave the region
  std::map<const Value*, std::vector<ValuePtr>> leaves;  // canonical value -> the values to store
  for (const Node& n : nodes) {
    const ValuePtr& v = prog_->ops[n.op].result;
    bool outside = outputs_.count(v.get()) > 0;
    const auto uit = users_.find(v.get());
    if (uit != users_.end())
      for (size_t u : uit->second) outside = outside || !members.count(u);
    if (outside) leaves[canon(v)].push_back(v);
  }
  // (an operation list whose intermediate values are wanted outside as well stays apart, as a visible softmax does)
  for (const Node& n : nodes)
    for (const ValuePtr& v : {n.a, n.b})
      if (v && leaves.count(canon(v))) return false;
  // emission: vector slots by last use
  Step s;
  s.kind = Step::Rows;
  pml_hip_rows_desc& d = s.rows;
  d.dtype = hipType(dt);
  d.cols = shape.sizes[r - 1];
  d.rows = rowsOf(shape);
  std::map<const Value*, size_t> last;
  for (size_t k = 0; k < nodes.size(); ++k) {
    if (nodes[k].opcode == -1) continue;
    last[canon(nodes[k].a)] = k;
    if (nodes[k].b) last[canon(nodes[k].b)] = k;
  }
  std::map<const Value*, int> slot, scalar, input;
  std::vector<bool> vec_busy(PML_HIP_ROWS_VECTORS, false), sca_busy(PML_HIP_ROWS_SCALARS, false);
  std::vector<ValuePtr> inputs;
  bool fits = true;
  auto push = [&](const pml_hip_rows_step& st) {
    if (d.n_steps >= PML_HIP_ROWS_STEPS) {
      fits = false;
      return;
    }
    d.steps[d.n_steps++] = st;
  };
  auto take = [&](std::vector<bool>& busy) {
    for (size_t k = 0; k < busy.size(); ++k)
      if (!busy[k]) {
        busy[k] = true;
        return static_cast<int>(k);
      }
    fits = false;
    return 0;
  };
  auto inputIndex = [&](const ValuePtr& v) {
    const auto it = input.find(v.get());
    if (it != input.end()) return it->second;
    if (inputs.size() >= PML_HIP_ROWS_IO) {
      fits = false;
      return 0;
    }
    inputs.push_back(v);
    return input[v.get()] = static_cast<int>(inputs.size()) - 1;
  };
  // uses of an outside matrix: one that is read again is kept in a slot from its first use on
  std::map<const Value*, int> full_uses;
  for (const Node& n : nodes) {
    if (n.opcode == -1) continue;
    for (const ValuePtr& v : {n.a, n.b})
      if (v && !made.count(canon(v)) && isFull(v)) ++full_uses[v.get()];
  }
  auto operand = [&](const ValuePtr& v, int32_t* kind, int32_t* index) {
    const Value* c = canon(v);
    if (slot.count(c)) {
      *kind = PML_HIP_ROWS_VECTOR;
      *index = slot[c];
    } else if (scalar.count(c)) {
      *kind = PML_HIP_ROWS_SCALAR;
      *index = scalar[c];
    } else if (isFull(v)) {
      *kind = PML_HIP_ROWS_FULL;
      *index = inputIndex(v);
      if (full_uses[v.get()] > 1) {
        pml_hip_rows_step ld{};
        ld.kind = PML_HIP_ROWS_MAP;
        ld.a_kind = PML_HIP_ROWS_FULL;
        ld.a = *index;
        ld.dst = take(vec_busy);
        push(ld);
        slot[c] = ld.dst;
        d.n_vectors = std::max(d.n_vectors, ld.dst + 1);
        *kind = PML_HIP_ROWS_VECTOR;
        *index = ld.dst;
      }
    } else if (v->shape.elements() == 1) {
      *kind = PML_HIP_ROWS_ONE;
      *index = inputIndex(v);
    } else if (isRow(v)) {
      *kind = PML_HIP_ROWS_ROW;
      *index = inputIndex(v);
    } else {
      *kind = PML_HIP_ROWS_COLUMNS;
      *index = inputIndex(v);
    }
  };
  std::vector<ValuePtr> outs;
  for (size_t k = 0; k < nodes.size() && fits; ++k) {
    const Node& n = nodes[k];
    if (n.opcode == -1) continue;
    const ValuePtr& v = prog_->ops[n.op].result;
    pml_hip_rows_step st{};
    st.opcode = n.opcode;
    operand(n.a, &st.a_kind, &st.a);
    if (n.reduce) {
      st.kind = PML_HIP_ROWS_REDUCE;
      st.imm = static_cast<float>(n.imm_value);
    } else {
      if (n.imm) {
        st.b_kind = PML_HIP_ROWS_IMM;
        st.imm = static_cast<float>(n.imm_value);
      } else if (n.b) {
        operand(n.b, &st.b_kind, &st.b);
      }
      st.kind = n.row ? PML_HIP_ROWS_MAP_SCALAR : PML_HIP_ROWS_MAP;
    }
    // operands that end here give up their slots; a lane reads its columns before it writes them, so the result may take one
    for (const ValuePtr& o : {n.a, n.b})
      if (o && last[canon(o)] == k && !leaves.count(canon(o))) {
        if (slot.count(canon(o))) vec_busy[static_cast<size_t>(slot[canon(o)])] = false;
        if (scalar.count(canon(o))) sca_busy[static_cast<size_t>(scalar[canon(o)])] = false;
      }
    if (n.row) {
      st.dst = take(sca_busy);
      scalar[v.get()] = st.dst;
    } else {
      st.dst = take(vec_busy);
      slot[v.get()] = st.dst;
      d.n_vectors = std::max(d.n_vectors, st.dst + 1);
    }
    push(st);
    const auto leave = leaves.find(v.get());
    if (leave == leaves.end()) continue;
    for (const ValuePtr& to : leave->second) {
      if (outs.size() >= PML_HIP_ROWS_IO) {
        fits = false;
        break;
      }
      pml_hip_rows_step out{};
      out.kind = n.row ? PML_HIP_ROWS_STORE_SCALAR : PML_HIP_ROWS_STORE;
      out.a_kind = n.row ? PML_HIP_ROWS_SCALAR : PML_HIP_ROWS_VECTOR;
      out.a = st.dst;
      out.dst = static_cast<int>(outs.size());
      outs.push_back(to);
      push(out);
    }
    // (a stored value keeps its slot while later steps of the region read it)
    if (!last.count(v.get())) (n.row ? sca_busy : vec_busy)[static_cast<size_t>(st.dst)] = false;
  }
  d.n_in = static_cast<int32_t>(inputs.size());
  d.n_out = static_cast<int32_t>(outs.size());
  if (!fits || outs.empty() || !pml_hip_rows_takes(&d)) return false;
  for (const ValuePtr& v : inputs) s.operands.push_back(bufferFor(v));
  for (const ValuePtr& v : outs) s.outs.push_back(bufferFor(v));
  for (const Node& n : nodes) consumed_.insert(n.op);
  s.bytes = static_cast<double>(shape.getByteSize()) * 2;
  std::stringstream ss;
  ss << "row program " << util::mnemonic(dt) << " over the last axis of " << shape.str() << ": " << work << " operations, " << reductions << " of them reductions, "
     << d.n_steps << " steps, " << d.n_vectors << " vectors";
  for (const ValuePtr& v : outs) ss << " -> " << v->shape.str();
  s.text = ss.str();
  plan_->steps.push_back(s);
  return true;
}

}  // namespace pmlc::target::hip
