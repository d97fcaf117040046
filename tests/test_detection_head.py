"""The detection head taken from its maps in one launch (fx_head_nms, ext/detection_head.cpp): the same bits as the chain of
functors that a function built from host examples keeps."""
import ctypes
from typing import List, Tuple

import pytest
import torch
from torch import Tensor

import functs_amd.jit as fj
from functs_amd import _C, _lib, aot
from functs_amd.benchmark import PROGRAMS
from functs_amd.benchmark.inputs import yolov3_head
from functs_amd.benchmark.programs import _decode_stack, _yolov3_head_scores


def no_threshold(pred_maps: List[Tensor], base_anchors: List[Tensor]):
    """Every class of every kept row is a candidate."""
    bboxes, cls_scores, objectness = _yolov3_head_scores(pred_maps, base_anchors)
    det_results: List[Tuple[Tensor, Tensor]] = []
    for i in range(bboxes.size(0)):
        o = objectness[i]
        keep = o >= 0.4
        det_results.append(torch.ops.functs.multiclass_nms(bboxes[i][keep, :], cls_scores[i][keep, :], o[keep], 0.0, 0.45, 100, True))
    return det_results


def strict(pred_maps: List[Tensor], base_anchors: List[Tensor]):
    """Only a score that rounds to 1 passes, more results than candidates."""
    bboxes, cls_scores, objectness = _yolov3_head_scores(pred_maps, base_anchors)
    det_results: List[Tuple[Tensor, Tensor]] = []
    for i in range(bboxes.size(0)):
        o = objectness[i]
        keep = o >= 0.4
        det_results.append(torch.ops.functs.multiclass_nms(bboxes[i][keep, :], cls_scores[i][keep, :], o[keep], 0.99999994, 0.3, 300, True))
    return det_results


def scaled(pred_maps: List[Tensor], base_anchors: List[Tensor]):
    """Does more with the detections than to list them."""
    bboxes, cls_scores, objectness = _yolov3_head_scores(pred_maps, base_anchors)
    out: List[Tensor] = []
    for i in range(bboxes.size(0)):
        o = objectness[i]
        keep = o >= 0.005
        dets, labels = torch.ops.functs.multiclass_nms(bboxes[i][keep, :], cls_scores[i][keep, :], o[keep], 0.05, 0.45, 100, True)
        out.append(dets * 0.5)
    return out


def _given(pred_maps: List[Tensor], base_anchors: List[Tensor], shifts: List[Tensor], strides: Tensor):
    """The head with its tables as arguments (types of what a program makes on a GPU are not known without one)."""
    num_imgs = pred_maps[0].size(0)
    num_attrib = pred_maps[0].size(1) // base_anchors[0].size(0)
    mlvl_anchors: List[Tensor] = []
    flatten_preds: List[Tensor] = []
    for lvl in range(3):
        mlvl_anchors.append((base_anchors[lvl].unsqueeze(0) + shifts[lvl]).reshape(-1, 4))
        pred = pred_maps[lvl].permute(0, 2, 3, 1).reshape(num_imgs, -1, num_attrib).clone()
        pred[..., :2].sigmoid_()
        flatten_preds.append(pred.clone())
    preds = torch.cat(flatten_preds, dim=1)
    bboxes = _decode_stack(torch.cat(mlvl_anchors), preds[..., :4], strides)
    padding = bboxes.new_zeros(num_imgs, bboxes.size(1), 1)
    return bboxes, torch.cat([preds[..., 5:].sigmoid(), padding], dim=-1), preds[..., 4].sigmoid()


def _given_tail(bboxes: Tensor, cls_scores: Tensor, objectness: Tensor):
    det_results: List[Tuple[Tensor, Tensor]] = []
    for i in range(bboxes.size(0)):
        o = objectness[i]
        keep = o >= 0.005
        det_results.append(torch.ops.functs.multiclass_nms(bboxes[i][keep, :], cls_scores[i][keep, :], o[keep], 0.05, 0.45, 100, True))
    return det_results


def only_read(pred_maps: List[Tensor], base_anchors: List[Tensor], shifts: List[Tensor], strides: Tensor):
    bboxes, cls_scores, objectness = _given(pred_maps, base_anchors, shifts, strides)
    return _given_tail(bboxes, cls_scores, objectness)


def written_before(pred_maps: List[Tensor], base_anchors: List[Tensor], shifts: List[Tensor], strides: Tensor):
    pred_maps[0].mul_(0.5)
    bboxes, cls_scores, objectness = _given(pred_maps, base_anchors, shifts, strides)
    return _given_tail(bboxes, cls_scores, objectness)


def written_behind(pred_maps: List[Tensor], base_anchors: List[Tensor], shifts: List[Tensor], strides: Tensor):
    bboxes, cls_scores, objectness = _given(pred_maps, base_anchors, shifts, strides)
    det_results = _given_tail(bboxes, cls_scores, objectness)
    pred_maps[0].zero_()
    return det_results


def map_written(pred_maps: List[Tensor], base_anchors: List[Tensor], shifts: List[Tensor], strides: Tensor):
    bboxes, cls_scores, objectness = _given(pred_maps, base_anchors, shifts, strides)
    pred_maps[0].zero_()
    return _given_tail(bboxes, cls_scores, objectness)


def anchors_written(pred_maps: List[Tensor], base_anchors: List[Tensor], shifts: List[Tensor], strides: Tensor):
    bboxes, cls_scores, objectness = _given(pred_maps, base_anchors, shifts, strides)
    base_anchors[1].zero_()
    return _given_tail(bboxes, cls_scores, objectness)


def strides_written(pred_maps: List[Tensor], base_anchors: List[Tensor], shifts: List[Tensor], strides: Tensor):
    bboxes, cls_scores, objectness = _given(pred_maps, base_anchors, shifts, strides)
    strides.zero_()
    return _given_tail(bboxes, cls_scores, objectness)


def _kinds(block):
    for n in block.nodes():
        yield n.kind()
        for b in n.blocks():
            yield from _kinds(b)


def _both(program, args):
    """(function with the one launch, function with the chain: its examples lie on the host), built for the same shapes"""
    gargs = [[t.cuda() for t in a] for a in args]
    one, chain = fj.build(fj.script(program), gargs), fj.build(fj.script(program), args)
    assert list(_kinds(one.graph.block())).count("fx::detection_head_pairs") == 1
    assert "fx::detection_head_pairs" not in list(_kinds(chain.graph.block()))
    return one, chain, gargs


def _launches(fn, args):
    before = aot.launch_stats()[0]
    out = fn(*args)
    torch.cuda.synchronize()
    return out, aot.launch_stats()[0] - before


def _assert_same(got, ref):
    assert len(got) == len(ref)
    for (d, l), (rd, rl) in zip(got, ref):
        assert torch.equal(l, rl) and torch.equal(d, rd)


def test_a_function_built_from_host_examples_keeps_the_chain():
    fn = fj.build(fj.script(PROGRAMS["yolo_head_nms"]), list(yolov3_head(0, 2, (2, 4, 8), 5)))
    assert not any("detection_head" in k for k in _kinds(fn.graph.block()))


WRITES = (map_written, anchors_written, strides_written)


@pytest.mark.parametrize("program", (only_read, written_before, written_behind) + WRITES)
def test_writes_between_the_head_and_its_tail_keep_the_chain(program):
    """The launch and the chain beside it stand at the tail: what the program writes before that, they would read."""
    def hint(*sizes):
        return torch.TensorType.get().with_dtype(torch.float32).with_sizes(list(sizes)).with_device(torch.device("cuda", 0))
    grids = (2, 4, 8)
    g = fj.script(program).graph.copy()
    _C._jit_pass_fait_pipeline(g, [torch.TupleType([hint(2, 30, f, f) for f in grids]), torch.TupleType([hint(3, 4) for f in grids]),
                                   torch.TupleType([hint(f * f, 1, 4) for f in grids]), hint(252, 1)])
    before = list(g.nodes())
    order = [n.kind() for n in before]
    assert _C._jit_pass_fuse_detection_head(g) == (program not in WRITES)
    if program in WRITES:
        assert [n.kind() for n in g.nodes()] == order
        write = next(k for k, kind in enumerate(order) if kind == "aten::copy_")
        assert order.index("tssa::ParallelFunctor") < write < order.index("functs::multiclass_nms_batched")


@pytest.mark.gpu
@pytest.mark.parametrize("program", (written_before, written_behind) + WRITES)
def test_writes_are_seen_where_the_program_makes_them(program):
    batch, grids, classes = 2, (4, 8, 16), 5
    maps, bases = yolov3_head(12, batch, grids, classes)
    shifts = [torch.rand(f * f, 1, 4) * 100.0 for f in grids]
    strides = torch.full((3 * sum(f * f for f in grids), 1), 8.0)

    def on_gpu():
        return [[t.cuda() for t in a] for a in (maps, bases, shifts)] + [strides.cuda()]
    print(program.__name__, flush=True)
    plain = fj.build(fj.script(only_read), on_gpu())
    args = on_gpu()
    if program is written_before:
        args[0][0].mul_(0.5)
    ref = plain(*args)
    fn, args = fj.build(fj.script(program), on_gpu()), on_gpu()
    _assert_same(fn(*args), ref)
    assert sum(d.size(0) for d, _ in ref) > 0
    same = [torch.equal(t, r) for a, b in zip(args, on_gpu()) for t, r in (zip(a, b) if isinstance(a, list) else [(a, b)])]
    assert same.count(False) == 1


# Runs of class scores that end inside a vector, inside a group of 256 and with one; one cell; up to 16 and one to three images
@pytest.mark.gpu
@pytest.mark.parametrize("batch,grids,classes", [(1, (1, 2, 3), 4), (3, (2, 4, 8), 5), (2, (4, 8, 16), 16), (16, (7, 14, 28), 10), (1, (13, 26, 52), 80),
                                                 (3, (19, 38, 76), 37), (300, (1, 2, 3), 4)])
def test_same_bits_as_the_chain(batch, grids, classes):
    args = list(yolov3_head(batch + classes, batch, grids, classes))
    for m in args[0]:
        m.view(batch, 3, 5 + classes, -1)[:, :, 5:] -= 1.0 if grids[0] < 4 else 3.5 if grids[0] < 8 else 6.0
    print("head", batch, grids, classes, flush=True)
    one, chain, gargs = _both(PROGRAMS["yolo_head_nms"], args)
    got, launches = _launches(one, gargs)
    ref, n_chain = _launches(chain, gargs)
    assert launches == 1 and n_chain > 1
    _assert_same(got, ref)
    assert sum(d.size(0) for d, _ in got) > 0


@pytest.mark.gpu
def test_other_thresholds_and_special_values():
    args = list(yolov3_head(3, 2, (3, 6, 12), 6))
    flat = args[0][2].view(2, 3, 11, 144)
    for k, x in enumerate((float("nan"), float("inf"), -float("inf"))):
        flat[:, k, 5, 3::7] = x          # class logits
        flat[:, k, 4, 5::11] = x         # objectness
    flat[0, 0, 0, 7] = flat[1, 2, 2, 9] = 95.0
    flat[:, 1, 7, 2::9] = 40.0           # scores that are 1
    for program in (no_threshold, strict, PROGRAMS["yolo_head_nms"]):
        print(program.__name__, flush=True)
        one, chain, gargs = _both(program, args)
        (got, n_one), (ref, n_chain) = _launches(one, gargs), _launches(chain, gargs)
        assert n_one == 1 and n_chain > 1
        _assert_same(got, ref)
        assert sum(d.size(0) for d, _ in got) > 0


@pytest.mark.gpu
def test_detections_that_are_used_otherwise():
    args = list(yolov3_head(6, 2, (4, 8, 16), 20))
    for m in args[0]:
        m.view(2, 3, 25, -1)[:, :, 5:] -= 4.0
    gargs = [[t.cuda() for t in a] for a in args]
    one, pairs = fj.build(fj.script(scaled), gargs), fj.build(fj.script(PROGRAMS["yolo_head_nms"]), gargs)
    assert list(_kinds(one.graph.block())).count("fx::detection_head") == 1
    got, ref = one(*gargs), pairs(*gargs)
    assert len(got) == len(ref) and all(torch.equal(d, rd * 0.5) for d, (rd, _) in zip(got, ref)) and sum(d.size(0) for d in got) > 0


@pytest.mark.gpu
def test_rows_that_are_not_kept_do_not_count_as_candidates():
    """More class scores of an image above the threshold than there is room for, of rows that the objectness drops: nothing is
    refused.  The same with rows that are kept is refused, and the next call works.  (A workgroup's share is not read again here: it is
    14 336 scores; test_shares_that_are_read_again.)"""
    args = list(yolov3_head(4, 1, (19, 38, 76), 80))
    for m in args[0]:
        v = m.view(1, 3, 85, -1)
        v[:, :, 5:] = v[:, :, 5:].abs()
        v[:, :, 4] = -9.0
        v[:, :, 4, 5::200] = 2.0         # 117 rows of 80 candidates
    one, chain, gargs = _both(PROGRAMS["yolo_head_nms"], args)
    print("again", flush=True)
    got, launches = _launches(one, gargs)
    assert launches == 1
    _assert_same(got, chain(*gargs))
    full = [[m.clone() for m in gargs[0]], gargs[1]]
    for m in full[0]:
        m.view(1, 3, 85, -1)[:, :, 4:] = 1.0
    print("refused", flush=True)
    with pytest.raises(RuntimeError, match="more than 16384 candidates"):
        one(*full)
    _assert_same(one(*gargs), got)


@pytest.mark.gpu
def test_operands_that_the_launch_does_not_take_run_the_chain():
    args = list(yolov3_head(5, 2, (4, 8, 16), 20))
    for m in args[0]:
        m.view(2, 3, 25, -1)[:, :, 5:] -= 4.0
    one, chain, gargs = _both(PROGRAMS["yolo_head_nms"], args)
    ref, n_chain = _launches(chain, gargs)
    assert n_chain > 1
    last = [[m.contiguous(memory_format=torch.channels_last) for m in gargs[0]], gargs[1]]
    print("channels last", flush=True)
    got, n = _launches(one, last)
    assert n == n_chain
    _assert_same(got, ref)
    grad = [[m.clone().requires_grad_() for m in gargs[0]], gargs[1]]
    print("gradients", flush=True)
    got, n = _launches(one, grad)
    assert n == n_chain
    _assert_same(got, ref)
    with torch.no_grad():
        got, n = _launches(one, grad)
    assert n == 1
    _assert_same(got, ref)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    print("another stream", flush=True)
    with torch.cuda.stream(side):
        got, n = _launches(one, gargs)
    assert n == 1
    _assert_same(got, ref)


def test_descriptors_that_do_not_fit_are_refused():
    """(nothing is launched: every descriptor is refused on the host)"""
    one = (ctypes.c_float * 4)()
    at = ctypes.cast(one, ctypes.c_void_p).value

    def call(levels=1, cells=4, anchors=3, rows=12, classes=5, max_num=10, cap=128, maps=at, mode=1):
        h = _lib.FxHeadDesc()
        h.n_levels, h.keep_thr, h.strides = levels, 0.1, at
        for k in range(4):
            h.maps[k], h.bases[k], h.shifts[k], h.cells[k], h.anchors[k] = maps, at, at, cells, anchors
        d = _lib.FxNmsDesc()
        d.mode, d.n_tasks, d.rows, d.n_classes, d.max_num, d.key_capacity = mode, 1, rows, classes, max_num, cap
        d.dets = d.out_labels = d.n_out = at
        return _lib.lib.fx_head_nms(ctypes.byref(h), ctypes.byref(d), None)

    for bad in (dict(levels=0), dict(levels=5), dict(cells=0, rows=0), dict(rows=11), dict(cells=1, rows=3, classes=3), dict(max_num=0), dict(max_num=1025),
                dict(cap=0), dict(cap=16385), dict(maps=None), dict(mode=0), dict(classes=0), dict(cells=1 << 20, rows=3 << 20, classes=1 << 10), dict()):
        assert call(**bad) < 0, bad


def _elements_of_workgroups(batch, grids, classes):
    """Class scores that every workgroup of an image scans (fx_launch_head_nms: groups of 256, none across two runs)."""
    groups = []
    for g in grids:
        run = classes * g * g
        groups += ([256] * (run // 256) + ([run % 256] if run % 256 else [])) * 3
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    slices = min(max(cus // batch, 1), 128, -(-len(groups) // 16))
    share = -(-len(groups) // slices)
    return [sum(groups[k * share:(k + 1) * share]) for k in range(slices)]


def _few_rows_kept(seed, batch, grids, classes, rows):
    """Every class score passes the threshold, the objectness of `rows` rows an image does."""
    g = torch.Generator().manual_seed(seed)
    args = list(yolov3_head(seed, batch, grids, classes))
    views = [m.view(batch, 3, 5 + classes, -1) for m in args[0]]
    starts = [0]
    for v in views:
        v[:, :, 5:].clamp_(-2.0, 2.0)
        v[:, :, 4] = -9.0
        starts.append(starts[-1] + 3 * v.size(3))
    for b in range(batch):
        for row in torch.randperm(starts[-1], generator=g)[:rows].tolist():
            level = max(k for k in range(len(views)) if row >= starts[k])
            r = row - starts[level]
            views[level][b, r // views[level].size(3), 4, r % views[level].size(3)] = 2.0
    return args


# Workgroups with more class scores above the threshold than the 2 048 whose boxes LDS holds, up to 16 384, of which few are
# left; alone with their image and several to one.  Few, 700 and just up to 2 048 candidates (ordered by buckets), more (sorted).
@pytest.mark.gpu
@pytest.mark.parametrize("batch,grids,classes,rows,elements", [
    (1, (3, 6, 12), 5, (1, 140, 409, 410), 2835), (130, (4, 8, 16), 8, (1, 88, 256, 257), 8064), (130, (4, 8, 16), 16, (1, 43, 128, 129), 16128),
    (8, (19, 38, 76), 10, (1, 70, 204, 205), 7168), (1, (19, 38, 76), 80, (1, 9, 25, 26), 14336), (2, (19, 38, 76), 64, (1, 11, 32, 33), 11520)])
def test_few_candidates_of_many_scores_above_the_threshold(batch, grids, classes, rows, elements):
    fullest = max(_elements_of_workgroups(batch, grids, classes))
    assert 2048 < fullest <= 16384 and fullest == elements
    one = None
    for kept in rows:
        args = _few_rows_kept(kept, batch, grids, classes, kept)
        print("few of many", batch, grids, classes, kept, flush=True)
        if one is None:
            one, chain, _ = _both(PROGRAMS["yolo_head_nms"], args)
        gargs = [[t.cuda() for t in a] for a in args]
        (got, launches), (ref, n_chain) = _launches(one, gargs), _launches(chain, gargs)
        assert launches == 1 and n_chain > 1
        _assert_same(got, ref)
        assert min(d.size(0) for d, _ in got) > 0


def below_zero(pred_maps: List[Tensor], base_anchors: List[Tensor]):
    """Every number is a score above the threshold."""
    bboxes, cls_scores, objectness = _yolov3_head_scores(pred_maps, base_anchors)
    det_results: List[Tuple[Tensor, Tensor]] = []
    for i in range(bboxes.size(0)):
        o = objectness[i]
        keep = o >= 0.4
        det_results.append(torch.ops.functs.multiclass_nms(bboxes[i][keep, :], cls_scores[i][keep, :], o[keep], -0.5, 0.45, 1000, True))
    return det_results


@pytest.mark.gpu
def test_scores_of_zero_above_a_threshold_below_zero():
    """(a class that is masked out: its logit is -inf, its score 0)"""
    args = list(yolov3_head(8, 2, (2, 4, 8), 6))
    for m in args[0]:
        m.view(2, 3, 11, -1)[:, :, 6::2] = -float("inf")
    print("below zero", flush=True)
    one, chain, gargs = _both(below_zero, args)
    (got, n_one), (ref, n_chain) = _launches(one, gargs), _launches(chain, gargs)
    assert n_one == 1 and n_chain > 1
    assert all(bool((d[:, 4] == 0).any()) for d, _ in ref)
    _assert_same(got, ref)


def _refusal(fill):
    """The error of a descriptor of one level, and its message (nothing is launched: there is no workspace)."""
    at = ctypes.cast((ctypes.c_float * 4)(), ctypes.c_void_p).value
    h, d = _lib.FxHeadDesc(), _lib.FxNmsDesc()
    h.n_levels, h.keep_thr, h.strides = 1, 0.1, at
    h.maps[0], h.bases[0], h.shifts[0] = at, at, at
    d.mode, d.n_tasks, d.max_num, d.key_capacity = 1, 1, 10, 128
    d.dets = d.out_labels = d.n_out = at
    fill(h, d)
    return _lib.lib.fx_head_nms(ctypes.byref(h), ctypes.byref(d), None), _lib.lib.fx_last_error().decode()


# Class scores are numbered with every run rounded up to 256: runs of four are 64 times as many numbers as scores
@pytest.mark.parametrize("anchors,cells,classes,error", [(1 << 24, 1, 4, "workspace"), ((1 << 24) + 1, 1, 4, "beyond 32 bits"),
                                                         (1 << 24, 2, 50, "workspace"), ((1 << 24) + 1, 2, 50, "beyond 32 bits")])
def test_numbers_beyond_32_bits_are_refused(anchors, cells, classes, error):
    def fill(h, d):
        h.cells[0], h.anchors[0] = cells, anchors
        d.rows, d.n_classes = anchors * cells, classes
    rc, message = _refusal(fill)
    assert rc < 0 and error in message, message


@pytest.mark.gpu
def test_numbers_beyond_32_bits_run_the_chain():
    """(asked only, nothing is launched)"""
    fits = torch._C._jit_get_operation("fx::detection_head_fits")
    fits = fits[0] if isinstance(fits, tuple) else fits
    for anchors in (1 << 24, (1 << 24) + 1):
        maps, bases, shift, strides = (torch.empty(s, device="cuda") for s in ((1, anchors * 9, 1, 1), (anchors, 4), (1, 1, 4), (anchors, 1)))
        print("fits", anchors, flush=True)
        assert fits([maps], [bases], [shift], strides, 1, 4, 0.5, 0.05, 0.45, 100) == (anchors <= 1 << 24)


@pytest.mark.gpu
@pytest.mark.parametrize("shift", [4.0, 0.0])   # ordered by buckets, and sorted, where boxes are looked up by their rows
def test_a_row_stride_of_the_scores_is_not_read(shift):
    batch, grids, classes, max_num, cap = 2, (4, 8, 16), 5, 100, 16384
    maps, bases = yolov3_head(21, batch, grids, classes)
    for m in maps:
        m.view(batch, 3, 5 + classes, -1)[:, :, 5:] -= shift
    rows = 3 * sum(f * f for f in grids)
    maps, bases = [m.cuda() for m in maps], [b.cuda() for b in bases]
    shifts = [(torch.rand(f * f, 4, generator=torch.Generator().manual_seed(f)) * 100.0).cuda() for f in grids]
    strides = torch.full((rows,), 8.0, device="cuda")
    size = _lib.lib.fx_sort_nms_workspace_bytes(batch, cap)
    results = []
    for stride in (0, classes + 1):
        dets, labels = torch.full((batch, max_num, 5), -1.0, device="cuda"), torch.full((batch, max_num), -1, device="cuda")
        index, n, ws = torch.full_like(labels, -1), torch.full((batch,), -1, dtype=torch.int32, device="cuda"), torch.zeros(size, dtype=torch.uint8, device="cuda")
        h, d = _lib.FxHeadDesc(), _lib.FxNmsDesc()
        h.n_levels, h.keep_thr, h.strides = 3, 0.005, strides.data_ptr()
        for k, f in enumerate(grids):
            h.maps[k], h.bases[k], h.shifts[k], h.cells[k], h.anchors[k] = maps[k].data_ptr(), bases[k].data_ptr(), shifts[k].data_ptr(), f * f, 3
        d.mode, d.n_tasks, d.rows, d.n_classes, d.scores_row_stride = 1, batch, rows, classes, stride
        d.score_thr, d.iou_thr, d.max_num, d.key_capacity = 0.05, 0.45, max_num, cap
        d.dets, d.out_labels, d.out_index, d.n_out = dets.data_ptr(), labels.data_ptr(), index.data_ptr(), n.data_ptr()
        d.workspace, d.workspace_bytes = ws.data_ptr(), size
        print("stride", shift, stride, flush=True)
        assert _lib.lib.fx_head_nms(ctypes.byref(h), ctypes.byref(d), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        torch.cuda.synchronize()
        results.append([dets, labels, index, n])
    assert int(results[0][3].min()) > 0 and (shift > 0.0) == (sum(int((m.view(batch, 3, 5 + classes, -1)[:, :, 5:] > -2.944).sum()) for m in maps) < 2048 * batch)
    for a, b in zip(*results):
        assert torch.equal(a, b)


# More class scores above the threshold in a workgroup than its list has room for (16 384): its share is read again, with the
# objectness.  Several workgroups to an image, and one; ordered by buckets, and sorted.
@pytest.mark.gpu
@pytest.mark.parametrize("batch,grids,classes,rows,elements", [(4, (19, 38, 76), 80, (1, 25, 26, 200), 28672), (130, (4, 8, 16), 20, (1, 102, 103, 800), 20160)])
def test_shares_that_are_read_again(batch, grids, classes, rows, elements):
    assert max(_elements_of_workgroups(batch, grids, classes)) == elements > 16384
    one = None
    for kept in rows:
        args = _few_rows_kept(kept, batch, grids, classes, kept)
        print("read again", batch, grids, classes, kept, flush=True)
        if one is None:
            one, chain, _ = _both(PROGRAMS["yolo_head_nms"], args)
        gargs = [[t.cuda() for t in a] for a in args]
        (got, launches), (ref, n_chain) = _launches(one, gargs), _launches(chain, gargs)
        assert launches == 1 and n_chain > 1
        _assert_same(got, ref)
        assert min(d.size(0) for d, _ in got) > 0
