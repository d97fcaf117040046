// CollapseAttentionLoops: a decoding loop of single-query attention over a growing key / value
// cache, whose iterations carry the query, both caches and the position, becomes ONE node
// fx::attention_steps, which ToParallelFunctor wraps into a tssa::ParallelFunctor that runs the
// kernel fx_attention_steps.  (The reference leaves such a loop to the host: it carries values,
// fait/passes/parallelize_loops.cpp:17, and its trip count is no constant, unroll_loops.cpp:59-65.)
// The program recognised is the reference's functs/benchmark/simpleops/attention/attention.py:38-58
// after functionalization:
//
//   for i in range(n):                              prim::Loop carrying x, gen, k, v
//     k = select_rev(k, reshape(matmul(x, wk), [B, H, D]), 2, gen)     (through full slices)
//     v = select_rev(v, reshape(matmul(x, wv), [B, H, D]), 2, gen)
//     s = transpose(matmul(k, transpose(matmul(x, wq), 2, 3)), 2, 3)
//     x = matmul(matmul(softmax(s * scale, 3), v), wo)
//     gen = gen + 1
//
// The match is structural (order of the carried values free) and complete: a body with any other
// node is left alone, and so are operands without static shapes that fit the kernel or whose
// example did not lie on a GPU, where alone the kernel runs.
#include <torch/csrc/jit/ir/constants.h>

#include <limits>
#include <unordered_set>

#include "../../../include/fxhip.h"
#include "passes.h"
#include "symbols.h"

namespace functs {
using namespace torch::jit;

namespace {

bool isConst(Value* v, int64_t k) {
  auto c = toIValue(v);
  return c && c->isInt() && c->toInt() == k;
}
bool isTrue(Value* v) {
  auto c = toIValue(v);
  return c && c->isBool() && c->toBool();
}
// a dimension of a tensor of `rank` dimensions as a constant, counted from the front or the back
bool isDim(Value* v, int64_t dim, int64_t rank) { return isConst(v, dim) || isConst(v, dim - rank); }

struct AttnLoop {
  size_t x_i = 0, gen_i = 0, k_i = 0, v_i = 0;   // positions among the carried values
  Value *wq = nullptr, *wk = nullptr, *wv = nullptr, *wo = nullptr;
  double scale = 0.0;
};

struct Matcher {
  std::unordered_set<Node*> used;

  Node* is(Value* v, Symbol kind, size_t n_inputs) {
    Node* n = v->node();
    if (n->kind() != kind || n->inputs().size() != n_inputs || n->outputs().size() != 1) return nullptr;
    used.insert(n);
    return n;
  }
  // matmul(a, b): b for a given a
  Value* matmulBy(Value* v, Value* a) {
    Node* n = is(v, c10::aten::matmul, 2);
    return n && n->input(0) == a ? n->input(1) : nullptr;
  }
  // transpose of the last two of four dimensions: its operand
  Value* swapped(Value* v) {
    Node* n = is(v, c10::aten::transpose, 3);
    if (!n) return nullptr;
    const bool ok = (isDim(n->input(1), 2, 4) && isDim(n->input(2), 3, 4)) || (isDim(n->input(1), 3, 4) && isDim(n->input(2), 2, 4));
    return ok ? n->input(0) : nullptr;
  }
  bool fullRange(Value* start, Value* end, Value* step) {
    auto e = toIValue(end);
    return (start->mustBeNone() || isConst(start, 0)) &&
           (end->mustBeNone() || (e && e->isInt() && e->toInt() == std::numeric_limits<int64_t>::max())) && isConst(step, 1);
  }
  // slice_rev(self, src, dim, <everything>): src, for a self that is `self` or a select at `gen` of it
  Value* throughSliceRev(Value* v, Value* self, Value* gen) {
    while (v->node()->kind() == sym::SliceRev()) {
      Node* n = is(v, sym::SliceRev(), 6);
      if (!n || !fullRange(n->input(3), n->input(4), n->input(5))) return nullptr;
      if (n->input(0) != self) {
        Node* s = n->input(0)->node();
        if ((s->kind() != c10::aten::select && s->kind() != sym::Select()) || s->inputs().size() != 3 || s->input(0) != self ||
            !isDim(s->input(1), 2, 4) || s->input(2) != gen)
          return nullptr;
        used.insert(s);
      }
      v = n->input(1);
    }
    return v;
  }
  // the cache with row `gen` replaced by reshape(matmul(x, w), sizes): w
  Value* rowWrite(Value* v, Value* cache, Value* gen, Value* x, const std::vector<int64_t>& sizes) {
    v = throughSliceRev(v, cache, gen);
    Node* rev = v ? is(v, sym::SelectRev(), 4) : nullptr;
    if (!rev || rev->input(0) != cache || !isDim(rev->input(2), 2, 4) || rev->input(3) != gen) return nullptr;
    v = throughSliceRev(rev->input(1), cache, gen);
    if (!v) return nullptr;
    Node* n = v->node();
    if ((n->kind() != sym::Reshape() && n->kind() != sym::View() && n->kind() != c10::aten::reshape && n->kind() != c10::aten::view) ||
        n->inputs().size() != 2)
      return nullptr;
    used.insert(n);
    return sizesAre(n->input(1), sizes, x) ? matmulBy(n->input(0), x) : nullptr;
  }
  // the list [B, H, D]: a constant, or constants and the sizes of x (which keeps its own from step to step)
  bool sizesAre(Value* list, const std::vector<int64_t>& sizes, Value* x) {
    if (auto c = toIValue(list)) return c->isIntList() && c->toIntVector() == sizes;
    Node* n = list->node();
    if (n->kind() != c10::prim::ListConstruct || n->inputs().size() != sizes.size()) return false;
    used.insert(n);
    for (size_t i = 0; i < sizes.size(); ++i) {
      if (isConst(n->input(i), sizes[i])) continue;
      Node* size = is(n->input(i), c10::aten::size, 2);
      if (!size || size->input(0) != x || !isDim(size->input(1), i < 2 ? (int64_t)i : 3, 4)) return false;
    }
    return true;
  }
};

std::optional<std::vector<int64_t>> gpuFloatSizes(Value* v) {
  auto tt = v->type()->cast<c10::TensorType>();
  if (!tt || !tt->scalarType() || *tt->scalarType() != c10::kFloat || !tt->device() || !tt->device()->is_cuda()) return std::nullopt;
  return tt->sizes().concrete_sizes();
}

bool definedOutside(Value* v, Node* loop) {
  for (Block* b = v->node()->owningBlock(); b; b = b->owningNode() ? b->owningNode()->owningBlock() : nullptr)
    if (b->owningNode() == loop) return false;
  return true;
}

bool matchLoop(Node* loop, AttnLoop* r) {
  if (loop->kind() != c10::prim::Loop || loop->inputs().size() != 6 || !isTrue(loop->input(1))) return false;
  Block* b = loop->blocks()[0];
  if (!isTrue(b->outputs()[0])) return false;
  Matcher m;
  // the position, and x: the one tensor that ends in a product
  int gen = -1, x = -1, c0 = -1, c1 = -1;
  for (int i = 0; i < 4; ++i) {
    Value *p = b->inputs()[1 + i], *o = b->outputs()[1 + i];
    if (p->type()->kind() == c10::TypeKind::IntType) {
      Node* n = gen < 0 ? m.is(o, c10::aten::add, 2) : nullptr;
      if (!n || !((n->input(0) == p && isConst(n->input(1), 1)) || (n->input(1) == p && isConst(n->input(0), 1)))) return false;
      gen = i;
    } else if (o->node()->kind() == c10::aten::matmul && x < 0) {
      x = i;
    } else {
      (c0 < 0 ? c0 : c1) = i;
    }
  }
  if (gen < 0 || x < 0 || c0 < 0 || c1 < 0 || loop->output(gen)->hasUses()) return false;
  const auto xs = gpuFloatSizes(loop->input(2 + x)), cs0 = gpuFloatSizes(loop->input(2 + c0)), cs1 = gpuFloatSizes(loop->input(2 + c1));
  if (!xs || !cs0 || !cs1 || xs->size() != 4 || cs0->size() != 4 || *cs0 != *cs1) return false;
  const int64_t B = (*xs)[0], H = (*xs)[1], D = (*xs)[3], rows = (*cs0)[2];
  if ((*xs)[2] != 1 || *cs0 != std::vector<int64_t>{B, H, rows, D} || D > INT32_MAX || rows > INT32_MAX ||
      !fx_attention_steps_fits((int)D, (int)rows))
    return false;

  Value *px = b->inputs()[1 + x], *pg = b->inputs()[1 + gen];
  // x = matmul(matmul(softmax(transpose(matmul(k, transpose(matmul(x, wq)))) * scale), v), wo)
  Node* last = m.is(b->outputs()[1 + x], c10::aten::matmul, 2);
  Node* pv = last ? m.is(last->input(0), c10::aten::matmul, 2) : nullptr;
  Node* sm = pv ? m.is(pv->input(0), c10::aten::softmax, 3) : nullptr;
  if (!sm || !isDim(sm->input(1), 3, 4) || !sm->input(2)->mustBeNone()) return false;
  Node* mul = m.is(sm->input(0), c10::aten::mul, 2);
  auto scale = mul ? toIValue(mul->input(1)) : std::nullopt;
  if (!scale || !(scale->isDouble() || scale->isInt())) return false;
  Value* s = m.swapped(mul->input(0));
  Node* qk = s ? m.is(s, c10::aten::matmul, 2) : nullptr;
  Value* q = qk ? m.swapped(qk->input(1)) : nullptr;
  r->wq = q ? m.matmulBy(q, px) : nullptr;
  if (!r->wq) return false;
  r->wo = last->input(1);
  int k = -1, v = -1;
  for (int i : {c0, c1}) {
    if (b->outputs()[1 + i] == qk->input(0)) k = i;
    else if (b->outputs()[1 + i] == pv->input(1)) v = i;
  }
  if (k < 0 || v < 0) return false;
  const std::vector<int64_t> row{B, H, D}, weight{H, D, D};
  r->wk = m.rowWrite(b->outputs()[1 + k], b->inputs()[1 + k], pg, px, row);
  r->wv = r->wk ? m.rowWrite(b->outputs()[1 + v], b->inputs()[1 + v], pg, px, row) : nullptr;
  if (!r->wv) return false;
  for (Node* n : b->nodes())
    if (n->kind() != c10::prim::Constant && !m.used.count(n)) return false;
  for (Value* w : {r->wq, r->wk, r->wv, r->wo}) {
    const auto ws = gpuFloatSizes(w);
    if (!ws || *ws != weight || !definedOutside(w, loop)) return false;
  }
  r->scale = scale->toScalar().toDouble();
  r->x_i = (size_t)x; r->gen_i = (size_t)gen; r->k_i = (size_t)k; r->v_i = (size_t)v;
  return true;
}

// `cache` is add(t, number): t, and the number as a constant; the kernel adds it as it reads t
Value* addedTo(Value* cache, std::optional<double>* number) {
  Node* n = cache->node();
  if (n->kind() != c10::aten::add || n->inputs().size() != 3 || !isConst(n->input(2), 1)) return cache;
  auto c = toIValue(n->input(1));
  if (!c || !(c->isDouble() || c->isInt()) || gpuFloatSizes(n->input(0)) != gpuFloatSizes(cache)) return cache;
  *number = c->toScalar().toDouble();
  return n->input(0);
}

// one loop of the block or of a block inside it; false when there is none left
bool collapseOne(Block* b) {
  for (Node* n : b->nodes()) {
    AttnLoop r;
    if (!matchLoop(n, &r)) {
      for (Block* inner : n->blocks())
        if (collapseOne(inner)) return true;
      continue;
    }
    Graph* g = b->owningGraph();
    WithInsertPoint at(n);
    std::optional<double> k_add, v_add;
    Value *k = addedTo(n->input(2 + r.k_i), &k_add), *v = addedTo(n->input(2 + r.v_i), &v_add);
    auto optional = [&](const std::optional<double>& d) { return d ? g->insertConstant(*d) : g->insertConstant(c10::IValue()); };
    // the steps end at row `stop`: what the program subtracts the first row from, where it does
    Value *start = n->input(2 + r.gen_i), *trips = n->input(0), *stop = nullptr;
    if (trips->node()->kind() == c10::aten::sub && trips->node()->inputs().size() == 2 && trips->node()->input(1) == start)
      stop = trips->node()->input(0);
    else
      stop = g->insert(c10::aten::add, {start, trips});
    Node* a = g->create(sym::AttentionSteps(), {n->input(2 + r.x_i), k, v, r.wq, r.wk, r.wv, r.wo, start, stop, g->insertConstant(r.scale), optional(k_add), optional(v_add)}, 3);
    a->setSourceRange(n->sourceRange());
    a->insertBefore(n);
    const size_t carried[3] = {r.k_i, r.v_i, r.x_i};
    for (size_t o = 0; o < 3; ++o) {
      a->output(o)->copyMetadata(n->output(carried[o]));
      n->output(carried[o])->replaceAllUsesWith(a->output(o));
      // the results are new tensors: a copy that is their only use is left out
      const auto uses = a->output(o)->uses();
      if (uses.size() != 1 || uses[0].user->kind() != c10::aten::clone || !uses[0].user->input(1)->mustBeNone()) continue;
      uses[0].user->output()->replaceAllUsesWith(a->output(o));
      uses[0].user->destroy();
    }
    n->destroy();
    return true;
  }
  return false;
}

}  // namespace

bool CollapseAttentionLoops(std::shared_ptr<Graph> graph) {
  bool changed = false;
  while (collapseOne(graph->block())) changed = true;
  return changed;
}

}  // namespace functs
