// FuseDetectionHead: the chain that a YOLO-style detection head with its tail becomes,
//   functor (maps -> rows [B, N, 5 + C], boxes [B, N, 4])
//     -> compacting map functor (objectness filter, one task an image) -> functs::multiclass_nms_batched,
// gets ONE launch beside it, fx_head_nms, that takes its candidates from the maps themselves.  The rows and boxes of
// the chain exist for the tail alone, which looks at a few hundred of them: four 608 x 608 images of 80 classes move 125 MB
// through memory there, and read 31 MB here.  The program recognised is the reference's
// functs/benchmark/ai_model/yolov3/yolov3_bbox.py:12-23, 78-101, 194-243 as the passes before this one leave it:
//
//   level l:  pred = slice_rev(p, sigmoid(p[..., :2]), ..., :2),  p = reshape(permute(map_l, (0, 2, 3, 1)), [B, -1, 5 + C])
//             anchors_l = reshape(unsqueeze(base_l, 0) + shift_l, [-1, 4])          shift_l [cells, 1, 4]
//   preds = cat(pred_l, 1), anchors = cat(anchors_l)
//   boxes = stack of centre -/+ half size:  (a[:, :2] + a[:, 2:]) * 0.5 + (preds[..., :2] - 0.5) * strides,
//                                           (a[:, 2:] - a[:, :2]) * 0.5 * exp(preds[..., 2:4])
//   image i:  o = sigmoid(preds[..., 4])[i], kept rows o >= threshold, of boxes[i], cat(sigmoid(preds[..., 5:]), zeros)[i], o
//
// The match is structural and complete, as that of the loop kernels (attention.cpp).  Both forms stay in the graph, behind
//   if fx::detection_head_fits(operands): fx::detection_head(operands)  else: the chain,
// (fx::detection_head_pairs and the chain with its functs::unbatch_detection_pairs where that is all that is made of it)
// because a call may come with operands that only the chain serves (gradients, a capture, other devices).  They stand
// where the tail stood: a program that writes to the head's operands in between keeps the chain as it is.
#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/jit/ir/constants.h>
#include <torch/csrc/jit/runtime/custom_operator.h>

#include <limits>

#include "../../../include/fxhip.h"
#include "passes.h"
#include "symbols.h"

namespace functs {
using namespace torch::jit;

namespace {

bool isInt(Value* v, int64_t k) {
  auto c = toIValue(v);
  return c && c->isInt() && c->toInt() == k;
}
bool isNumber(Value* v, double k) {
  auto c = toIValue(v);
  return c && (c->isDouble() || c->isInt()) && c->toScalar().toDouble() == k;
}
bool isList(Value* v, const std::vector<int64_t>& want) {
  auto c = toIValue(v);
  return c && c->isIntList() && c->toIntVector() == want;
}
std::optional<std::vector<int64_t>> sizesOf(Value* v) {
  auto tt = v->type()->cast<c10::TensorType>();
  return tt ? tt->sizes().concrete_sizes() : std::nullopt;
}
bool floatOnGpu(Value* v) {
  auto tt = v->type()->cast<c10::TensorType>();
  return tt && tt->scalarType() && *tt->scalarType() == c10::kFloat && tt->device() && tt->device()->is_cuda();
}
Node* is(Value* v, Symbol kind, size_t n_inputs) {
  Node* n = v ? v->node() : nullptr;
  return n && n->kind() == kind && n->inputs().size() == n_inputs && n->outputs().size() == 1 ? n : nullptr;
}
Node* isEither(Value* v, Symbol a, Symbol b, size_t n_inputs) {
  Node* n = is(v, a, n_inputs);
  return n ? n : is(v, b, n_inputs);
}
Value* throughClones(Value* v) {
  while (v && v->node()->kind() == c10::aten::clone) v = v->node()->input(0);
  return v;
}
Value* unary(Value* v, Symbol kind) {
  Node* n = is(v, kind, 1);
  return n ? n->input(0) : nullptr;
}
// the last dimension of `of`, cut to [from, to) (to < 0: to its end); 0 and none are one start
bool lastDim(Value* dim, Value* of) {
  auto s = sizesOf(of);
  return isInt(dim, -1) || (s && isInt(dim, (int64_t)s->size() - 1));
}
bool boundIs(Value* v, int64_t k, bool open) {
  if (!open) return isInt(v, k);
  return v->mustBeNone() || isInt(v, k);
}
bool cutsLast(Node* n, size_t first, Value* of, int64_t from, int64_t to) {   // inputs first .. first + 3: dim, start, end, step
  return lastDim(n->input(first), of) && boundIs(n->input(first + 1), from, from == 0) &&
         (to < 0 ? n->input(first + 2)->mustBeNone() || isInt(n->input(first + 2), std::numeric_limits<int64_t>::max()) : isInt(n->input(first + 2), to)) &&
         isInt(n->input(first + 3), 1);
}
Value* lastSlice(Value* v, int64_t from, int64_t to) {
  Node* n = isEither(v, sym::Slice(), c10::aten::slice, 5);
  return n && cutsLast(n, 1, n->input(0), from, to) ? n->input(0) : nullptr;
}
Value* lastSelect(Value* v, int64_t at) {
  Node* n = isEither(v, sym::Select(), c10::aten::select, 3);
  return n && lastDim(n->input(1), n->input(0)) && isInt(n->input(2), at) ? n->input(0) : nullptr;
}
// a (op) b with weight 1
bool sum(Value* v, Symbol kind, Value** a, Value** b) {
  Node* n = is(v, kind, 3);
  if (!n || !isNumber(n->input(2), 1.0)) return false;
  *a = n->input(0);
  *b = n->input(1);
  return true;
}
Value* timesHalf(Value* v) {
  Node* n = is(v, c10::aten::mul, 2);
  return n && isNumber(n->input(1), 0.5) ? n->input(0) : nullptr;
}
std::vector<Value*> listItems(Value* v) {
  Node* n = v->node();
  return n->kind() == c10::prim::ListConstruct ? std::vector<Value*>(n->inputs().begin(), n->inputs().end()) : std::vector<Value*>{};
}
// the parts of a concatenation along `dim`; a value that is none is its one part
std::vector<Value*> parts(Value* v, int64_t dim) {
  Node* n = is(v, c10::aten::cat, 2);
  if (!n) return {v};
  return isInt(n->input(1), dim) ? listItems(n->input(0)) : std::vector<Value*>{};
}

struct Head {
  std::vector<Value*> maps, bases, shifts;   // in the functor's region
  Value* strides = nullptr;
  int64_t images = 0, rows = 0, classes = 0;
};

// the dense functor's region
bool matchDense(Graph& g, Value* preds, Value* boxes, Head* r) {
  auto ps = sizesOf(preds);
  if (!ps || ps->size() != 3 || (*ps)[2] < 6) return false;
  r->images = (*ps)[0];
  r->rows = (*ps)[1];
  r->classes = (*ps)[2] - 5;
  const int64_t width = (*ps)[2];
  // boxes
  Node* st = is(throughClones(boxes), c10::aten::stack, 2);
  if (!st || !(isInt(st->input(1), -1) || isInt(st->input(1), 2))) return false;
  const auto corner = listItems(st->input(0));
  if (corner.size() != 4) return false;
  Value *xy = nullptr, *wh = nullptr;
  for (int k = 0; k < 4; ++k) {
    Value *a = nullptr, *b = nullptr;
    if (!sum(corner[k], k < 2 ? c10::aten::sub : c10::aten::add, &a, &b)) return false;
    Value *c = lastSelect(a, k & 1), *s = lastSelect(b, k & 1);
    if (!c || !s || (xy && (c != xy || s != wh))) return false;
    xy = c;
    wh = s;
  }
  Value *centre = nullptr, *moved = nullptr, *lo = nullptr, *hi = nullptr;
  if (!sum(xy, c10::aten::add, &centre, &moved)) return false;
  Value* both = timesHalf(centre);
  if (!both || !sum(both, c10::aten::add, &lo, &hi)) return false;
  Value *anchors = lastSlice(lo, 0, 2), *bbox = nullptr;
  if (!anchors || lastSlice(hi, 2, -1) != anchors) return false;
  Node* mv = is(moved, c10::aten::mul, 2);
  Node* less = mv ? is(mv->input(0), c10::aten::sub, 3) : nullptr;
  if (!less || !isNumber(less->input(1), 0.5) || !isNumber(less->input(2), 1.0)) return false;
  r->strides = mv->input(1);
  bbox = lastSlice(less->input(0), 0, 2);
  if (!bbox || lastSlice(bbox, 0, 4) != preds) return false;
  Node* size = is(wh, c10::aten::mul, 2);
  Value* half = size ? timesHalf(size->input(0)) : nullptr;
  Value *hi2 = nullptr, *lo2 = nullptr;
  if (!half || !sum(half, c10::aten::sub, &hi2, &lo2) || lastSlice(hi2, 2, -1) != anchors || lastSlice(lo2, 0, 2) != anchors) return false;
  Value* e = unary(size->input(1), c10::aten::exp);
  if (!e || lastSlice(e, 2, -1) != bbox) return false;
  auto as = sizesOf(anchors), ss = sizesOf(r->strides);
  if (!as || *as != std::vector<int64_t>{r->rows, 4} || !ss || *ss != std::vector<int64_t>{r->rows, 1}) return false;
  // levels
  const auto level = parts(preds, 1), table = parts(anchors, 0);
  if (level.empty() || level.size() != table.size() || level.size() > FX_HEAD_LEVELS) return false;
  int64_t rows = 0;
  for (size_t l = 0; l < level.size(); ++l) {
    Node* rev = is(throughClones(level[l]), sym::SliceRev(), 6);
    if (!rev || !cutsLast(rev, 2, rev->input(0), 0, 2)) return false;
    Value* squashed = unary(rev->input(1), c10::aten::sigmoid);
    if (!squashed || lastSlice(squashed, 0, 2) != rev->input(0)) return false;
    Node* flat = isEither(throughClones(rev->input(0)), c10::aten::reshape, sym::Reshape(), 2);
    if (!flat || !(isList(flat->input(1), {r->images, -1, width}))) return false;
    Node* perm = isEither(flat->input(0), c10::aten::permute, sym::Permute(), 2);
    if (!perm || !isList(perm->input(1), {0, 2, 3, 1})) return false;
    Node* move = isEither(table[l], c10::aten::reshape, sym::Reshape(), 2);
    Value *base = nullptr, *shift = nullptr;
    if (!move || !isList(move->input(1), {-1, 4}) || !sum(move->input(0), c10::aten::add, &base, &shift)) return false;
    Node* un = isEither(base, c10::aten::unsqueeze, sym::Unsqueeze(), 2);
    if (!un || !isInt(un->input(1), 0)) return false;
    base = un->input(0);
    auto ms = sizesOf(perm->input(0)), bs = sizesOf(base), hs = sizesOf(shift);
    if (!ms || !bs || !hs || ms->size() != 4 || bs->size() != 2 || (*ms)[0] != r->images || (*bs)[1] != 4) return false;
    const int64_t cells = (*ms)[2] * (*ms)[3], anchors_l = (*bs)[0];
    if (anchors_l < 1 || cells < 1 || (*ms)[1] != anchors_l * width || *hs != std::vector<int64_t>{cells, 1, 4}) return false;
    rows += cells * anchors_l;
    r->maps.push_back(perm->input(0));
    r->bases.push_back(base);
    r->shifts.push_back(shift);
  }
  if (rows != r->rows) return false;
  for (const auto* vs : {&r->maps, &r->bases, &r->shifts})
    for (Value* v : *vs)
      if (v->node() != g.param_node() || !floatOnGpu(v)) return false;
  return r->strides->node() == g.param_node() && floatOnGpu(r->strides);
}

// the compacting functor's region: the sub-values behind the tail's boxes, scores and factors are those of the head
bool matchFilter(Graph& g, size_t boxes_o, size_t scores_o, size_t factors_o, const std::vector<int64_t>& preds_size, bool padded,
                 Value** preds, Value** boxes, double* keep_thr) {
  const auto outs = g.outputs();
  if (outs.size() != 4) return false;
  Value* index = g.inputs()[0];
  auto image = [&](Value* v) -> Value* {
    Node* n = isEither(v, c10::aten::select, sym::Select(), 3);
    return n && isInt(n->input(1), 0) && n->input(2) == index ? n->input(0) : nullptr;
  };
  Value* o = outs[factors_o];
  Node* keep = is(outs[3], c10::aten::ge, 2);
  auto thr = keep ? toIValue(keep->input(1)) : std::nullopt;
  if (!keep || keep->input(0) != o || !thr || !(thr->isDouble() || thr->isInt())) return false;
  *keep_thr = thr->toScalar().toDouble();
  Value* obj = image(o);
  obj = obj ? unary(obj, c10::aten::sigmoid) : nullptr;
  *preds = obj ? lastSelect(obj, 4) : nullptr;
  *boxes = image(outs[boxes_o]);
  Value* scores = image(outs[scores_o]);
  if (!*preds || !*boxes || !scores) return false;
  if (padded) {   // (what the last column holds does not matter, the tail cuts it off)
    Node* c = is(scores, c10::aten::cat, 2);
    const auto items = c ? listItems(c->input(0)) : std::vector<Value*>{};
    if (items.size() != 2 || !(isInt(c->input(1), -1) || isInt(c->input(1), 2))) return false;
    Node* z = items[1]->node();
    if (z->kind() != c10::aten::zeros || z->inputs().empty() || !isList(z->input(0), {preds_size[0], preds_size[1], 1})) return false;
    scores = items[0];
  }
  Value* cls = unary(scores, c10::aten::sigmoid);
  return cls && lastSlice(cls, 5, -1) == *preds && (*preds)->node() == g.param_node() && (*boxes)->node() == g.param_node();
}

// inputs of a functor and of its region: the region's first is the task's index
Value* argumentOf(Node* functor, Graph& g, Value* v) {
  for (size_t k = 1; k < g.inputs().size(); ++k)
    if (g.inputs()[k] == v) return functor->input(k - 1);
  return nullptr;
}
bool isFunctor(Node* n, bool map) {
  if (n->kind() != sym::ParallelFunctor() || (n->i(sym::is_parallel_map()) != 0) != map) return false;
  const bool compact = n->hasAttribute(sym::compact_rows()) && n->i(sym::compact_rows()) != 0;
  const bool padded = n->hasAttribute(sym::padded_outputs()) && n->i(sym::padded_outputs()) != 0;
  return compact == map && padded == map && n->g(c10::attr::Subgraph)->inputs().size() == n->inputs().size() + 1;
}

bool fuseAt(const std::shared_ptr<Graph>& graph, Node* tail) {
  static const Symbol batched = Symbol::fromQualString("functs::multiclass_nms_batched");
  if (tail->kind() != batched || tail->inputs().size() != 8) return false;
  Node* filter = tail->input(0)->node();
  if (!isFunctor(filter, true) || filter->outputs().size() != 4 || filter->owningBlock() != tail->owningBlock()) return false;
  size_t which[4];
  for (int k = 0; k < 4; ++k) {
    if (tail->input(k)->node() != filter || tail->input(k)->uses().size() != 1) return false;
    which[k] = tail->input(k)->offset();
  }
  if (which[3] != 3 || which[0] == which[1] || which[0] == which[2] || which[1] == which[2]) return false;
  for (int64_t p : filter->is(sym::is_parallel_args()))
    if (p != 0) return false;
  auto score_thr = toIValue(tail->input(4)), iou = toIValue(tail->input(5)), max_num = toIValue(tail->input(6)), padded = toIValue(tail->input(7));
  if (!score_thr || !iou || !max_num || !padded || !padded->isBool()) return false;

  const auto fg = filter->g(c10::attr::Subgraph);
  // the dense functor: what the filter's rows come from
  Node* dense = nullptr;
  for (Value* in : filter->inputs())
    if (in->node()->kind() == sym::ParallelFunctor()) {
      if (dense && in->node() != dense) return false;
      dense = in->node();
    }
  if (!dense || !isFunctor(dense, false) || dense->outputs().size() != 2 || dense->owningBlock() != tail->owningBlock()) return false;
  for (Value* o : dense->outputs())
    for (const Use& u : o->uses())
      if (u.user != filter) return false;
  const auto dg = dense->g(c10::attr::Subgraph);
  Value *f_preds = nullptr, *f_boxes = nullptr;
  double keep_thr = 0.0;
  // (sizes of the rows as the dense functor's results have them)
  for (size_t p = 0; p < 2; ++p) {
    auto ps = sizesOf(dg->outputs()[p]);
    Head h;
    if (!ps || ps->size() != 3 || !matchFilter(*fg, which[0], which[1], which[2], *ps, padded->toBool(), &f_preds, &f_boxes, &keep_thr)) continue;
    if (argumentOf(filter, *fg, f_preds) != dense->output(p) || argumentOf(filter, *fg, f_boxes) != dense->output(1 - p)) continue;
    if (!matchDense(*dg, dg->outputs()[p], dg->outputs()[1 - p], &h) || filter->i(sym::parallel_degree()) != h.images || h.images < 1) continue;
    // (the filter reads what the dense functor made, which nobody else has, and constants)
    if (writtenBetween(graph, dense, tail)) return false;

    Graph* g = graph.get();
    WithInsertPoint at(dense);
    auto tensors = [&](const std::vector<Value*>& vs) {
      std::vector<Value*> args;
      for (Value* v : vs) args.push_back(argumentOf(dense, *dg, v));
      Node* n = g->insertNode(g->createList(c10::TensorType::get(), args));
      return n->output();
    };
    std::vector<Value*> args{tensors(h.maps), tensors(h.bases), tensors(h.shifts), argumentOf(dense, *dg, h.strides), g->insertConstant(h.images),
                             g->insertConstant(h.classes), g->insertConstant(keep_thr), g->insertConstant(*score_thr), g->insertConstant(*iou),
                             g->insertConstant(*max_num)};
    Node* fits = g->insertNode(g->create(sym::DetectionHeadFits(), args, 1));
    fits->output()->setType(c10::BoolType::get());
    Node* choice = g->create(c10::prim::If, {fits->output()}, 0);
    choice->setSourceRange(tail->sourceRange());
    choice->insertBefore(tail);
    Block *yes = choice->addBlock(), *no = choice->addBlock();
    // where nothing but the list of pairs is made of the results, the launch waits for its own counts
    Node* pairs = tail->output(0)->uses().size() == 1 ? tail->output(0)->uses()[0].user : nullptr;
    const bool alone = pairs && pairs->kind() == Symbol::fromQualString("functs::unbatch_detection_pairs") && pairs->owningBlock() == tail->owningBlock() &&
                       pairs->inputs().size() == 3 && pairs->input(0) == tail->output(0) && pairs->input(1) == tail->output(1) &&
                       pairs->input(2) == tail->output(2) && tail->output(1)->uses().size() == 1 && tail->output(2)->uses().size() == 1;
    Node* end = alone ? pairs : tail;
    Node* head = g->create(alone ? sym::DetectionHeadPairs() : sym::DetectionHead(), args, end->outputs().size());
    head->setSourceRange(tail->sourceRange());
    yes->appendNode(head);
    for (size_t k = 0; k < end->outputs().size(); ++k) {
      head->output(k)->setType(end->output(k)->type());
      yes->registerOutput(head->output(k));
      Value* out = choice->addOutput()->setType(end->output(k)->type());
      end->output(k)->replaceAllUsesWith(out);
    }
    // the chain, in its order; what else feeds it is defined before it
    Node* last = nullptr;
    std::vector<Node*> chain{dense, filter, tail};
    if (alone) chain.push_back(pairs);
    for (Node* n : chain) {
      if (last) n->moveAfter(last);
      else {
        Node* mark = g->create(c10::prim::Constant, 0);
        no->appendNode(mark);
        n->moveAfter(mark);
        mark->destroy();
      }
      last = n;
    }
    for (Value* o : end->outputs()) no->registerOutput(o);
    return true;
  }
  return false;
}

bool fuseIn(const std::shared_ptr<Graph>& graph, Block* b) {
  // (collected first: what is joined moves nodes behind the tail into another block)
  bool changed = false;
  std::vector<Node*> tails;
  for (Node* n : b->nodes()) {
    for (Block* inner : n->blocks()) changed = fuseIn(graph, inner) || changed;
    if (n->kind() == Symbol::fromQualString("functs::multiclass_nms_batched")) tails.push_back(n);
  }
  for (Node* n : tails) changed = fuseAt(graph, n) || changed;
  return changed;
}

// --- the operators ----------------------------------------------------------------
struct Operands {
  std::vector<at::Tensor> maps, bases, shifts;
  at::Tensor strides;
  int64_t images, classes;
  double keep_thr, score_thr, iou;
  int64_t max_num;
};
Operands operandsOf(Stack& stack) {
  auto in = last(stack, 10);
  Operands o{in[0].toTensorVector(), in[1].toTensorVector(), in[2].toTensorVector(), in[3].toTensor(), in[4].toInt(), in[5].toInt(),
             in[6].toDouble(), in[7].toDouble(), in[8].toDouble(), in[9].toInt()};
  drop(stack, 10);
  return o;
}

// What the kernel serves; everything else is the chain's, with its own checks and errors.
bool fits(const Operands& o) {
  const size_t n = o.maps.size();
  if (n < 1 || n > FX_HEAD_LEVELS || o.bases.size() != n || o.shifts.size() != n || o.classes < 1 || o.max_num < 1 || o.max_num > FX_NMS_MAX_OUT) return false;
  const at::Tensor& first = o.maps[0];
  const int64_t width = 5 + o.classes;
  auto plain = [&](const at::Tensor& t) {
    return t.defined() && t.scalar_type() == at::kFloat && t.layout() == at::kStrided && t.is_cuda() && t.device() == first.device() &&
           t.is_contiguous() && !t.is_neg() && !(at::GradMode::is_enabled() && t.requires_grad()) && !t._fw_grad(0).defined() &&
           !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                                     c10::DispatchKey::Python, c10::DispatchKey::Functionalize}));
  };
  int64_t rows = 0, groups = 0;
  for (size_t l = 0; l < n; ++l) {
    const at::Tensor &m = o.maps[l], &b = o.bases[l], &s = o.shifts[l];
    if (!plain(m) || !plain(b) || !plain(s) || m.dim() != 4 || b.dim() != 2) return false;
    const int64_t anchors = b.size(0), cells = m.size(2) * m.size(3);
    if (m.size(0) != o.images || o.images < 1 || anchors < 1 || cells < 1 || b.size(1) != 4 || m.size(1) != anchors * width || s.numel() != cells * 4 ||
        cells * o.classes < 4 || m.numel() / o.images >= ((int64_t)1 << 31) || o.images * anchors >= ((int64_t)1 << 31))
      return false;
    rows += anchors * cells;
    groups += anchors * ((cells * o.classes + 255) / 256);
  }
  if (groups > (int64_t)FX_HEAD_MAX_GROUPS) return false;
  if (!plain(o.strides) || o.strides.numel() != rows || rows * width >= ((int64_t)1 << 31)) return false;
  if (at::autocast::is_autocast_enabled(at::kCUDA)) return false;
  // (a graph is left the chain, whose launches of a capture are known)
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(first.device().index()).stream(), &capture) != hipSuccess) (void)hipGetLastError();
  return capture == hipStreamCaptureStatusNone;
}

// what the launchers take besides the operands
struct Launch { fx_head_desc h; int64_t rows = 0; };
Launch launchOf(const Operands& o) {
  TORCH_CHECK(fits(o), "fx::detection_head: operands that the kernel does not serve");
  raiseAsyncErrors();
  Launch l;
  memset(&l.h, 0, sizeof l.h);
  l.h.n_levels = (int32_t)o.maps.size();
  l.h.keep_thr = (float)o.keep_thr;
  l.h.strides = o.strides.data_ptr<float>();
  for (size_t k = 0; k < o.maps.size(); ++k) {
    l.h.maps[k] = o.maps[k].data_ptr<float>();
    l.h.bases[k] = o.bases[k].data_ptr<float>();
    l.h.shifts[k] = o.shifts[k].data_ptr<float>();
    l.h.cells[k] = (uint32_t)(o.maps[k].size(2) * o.maps[k].size(3));
    l.h.anchors[k] = (uint32_t)o.bases[k].size(0);
    l.rows += (int64_t)l.h.cells[k] * l.h.anchors[k];
  }
  return l;
}
void runHead(Stack& stack) {
  const Operands o = operandsOf(stack);
  const Launch l = launchOf(o);
  auto r = launchHeadTail(l.h, o.maps[0].device(), o.images, l.rows, o.classes, o.score_thr, o.iou, o.max_num);
  for (at::Tensor& t : r) push(stack, std::move(t));
}
void runHeadPairs(Stack& stack) {
  const Operands o = operandsOf(stack);
  const Launch l = launchOf(o);
  push(stack, launchHeadPairs(l.h, o.maps[0].device(), o.images, l.rows, o.classes, o.score_thr, o.iou, o.max_num));
}

std::vector<c10::Argument> headArguments() {
  const auto list = c10::ListType::ofTensors();
  return {c10::Argument("maps", list), c10::Argument("bases", list), c10::Argument("shifts", list), c10::Argument("strides", c10::TensorType::get()),
          c10::Argument("images", c10::IntType::get()), c10::Argument("classes", c10::IntType::get()), c10::Argument("keep_thr", c10::FloatType::get()),
          c10::Argument("score_thr", c10::FloatType::get()), c10::Argument("iou_threshold", c10::FloatType::get()), c10::Argument("max_num", c10::IntType::get())};
}

// (all conservative: the answer of the first depends on modes and the current stream too)
RegisterOperators registerHead({
    Operator("fx::detection_head_fits", "", headArguments(), {c10::Argument("", c10::BoolType::get())},
             Operation([](Stack& stack) {
               const Operands o = operandsOf(stack);
               push(stack, fits(o));
             }),
             c10::AliasAnalysisKind::CONSERVATIVE),
    Operator("fx::detection_head", "", headArguments(),
             {c10::Argument("dets", c10::TensorType::get()), c10::Argument("labels", c10::TensorType::get()), c10::Argument("n", c10::TensorType::get())},
             Operation(runHead), c10::AliasAnalysisKind::CONSERVATIVE),
    Operator("fx::detection_head_pairs", "", headArguments(), {c10::Argument("", detectionPairsType())}, Operation(runHeadPairs),
             c10::AliasAnalysisKind::CONSERVATIVE),
});

}  // namespace

bool FuseDetectionHead(std::shared_ptr<Graph> graph) {
  const bool changed = fuseIn(graph, graph->block());
  if (changed) Validate(graph);
  return changed;
}

}  // namespace functs
