"""The TorchScript route: functs_amd.jit.script -> build (region formation ->
tssa::ParallelFunctor).  CPU tests check the graphs; the gpu tests run the built
functions on cuda:0 against stock TorchScript on the CPU (the oracle)."""
from typing import List

import pytest
import torch

import functs_amd.jit as fj
from functs_amd import _C
from oracle import configs as oc
from tests.util import assert_close, assert_exact, assert_boxes_close

SMALL_GRIDS = [2, 3, 4]


def _functors(graph):
    out = []

    def walk(block):
        for n in block.nodes():
            if n.kind() == "tssa::ParallelFunctor":
                out.append(n)
            for b in n.blocks():
                walk(b)

    walk(graph)
    return out


def _kinds(block, out=None):
    out = [] if out is None else out
    for n in block.nodes():
        out.append(n.kind())
        for b in n.blocks():
            _kinds(b, out)
    return out


def _built(name, args):
    return fj.build(fj.script(oc.CONFIGS[name][0]), list(args))


def test_c1_is_one_functor_with_a_collapsed_loop():
    args = oc.c1_inputs(0, 64)
    f = _built("c1", args)
    fs = _functors(f.graph)
    assert len(fs) == 1 and "prim::Loop" not in _kinds(f.graph)
    n = fs[0]
    assert n.i("is_parallel_map") == 0 and n.i("parallel_degree") == 1
    assert list(getattr(n, "is")("is_parallel_args")) == [1] * len(list(n.inputs()))
    sub = n.g("Subgraph")
    assert next(sub.inputs()).type().kind() == "NoneType"  # task-index placeholder (te_op.cpp:192)
    assert "fx::forall_select_rev" in _kinds(sub)


def test_c2_folds_the_row_mask_into_the_region():
    args = oc.c2_inputs(0, SMALL_GRIDS)
    f = _built("c2", args)
    fs = _functors(f.graph)
    assert len(fs) == 1
    assert fs[0].i("compact_rows") == 1
    assert "aten::index" not in _kinds(f.graph)
    sub = fs[0].g("Subgraph")
    assert len(list(sub.outputs())) == len(list(fs[0].outputs())) + 1  # mask rides last
    assert list(sub.outputs())[-1].node().kind() == "aten::ge"


def test_c5_is_one_parallel_map_functor():
    args = oc.c5_inputs(0, SMALL_GRIDS, 3)
    f = _built("c5", args)
    fs = _functors(f.graph)
    kinds = _kinds(f.graph)
    assert len(fs) == 1 and "prim::Loop" not in kinds and "aten::append" not in kinds
    n = fs[0]
    assert n.i("is_parallel_map") == 1 and n.i("compact_rows") == 1
    assert list(getattr(n, "is")("is_parallel_args")) == [0, 0, 0]  # preds, anchors, strides are shared
    sub = n.g("Subgraph")
    assert next(sub.inputs()).type().kind() == "IntType"  # the task index
    for o in n.outputs():
        assert o.type().kind() == "ListType"


def test_c3_is_decode_plus_class_map():
    """As in the reference the pipeline makes a dense functor (decode + softmax) and a class map;
    the last pass sinks the first into the second, because the library runs the merged region as
    one kernel (its size query on the scores becomes the constant of the static shape)."""
    args = oc.c3_inputs(0, 60, 7)
    _C._set_sink_producers(False)
    try:
        f = _built("c3", args)
    finally:
        _C._set_sink_producers(True)
    fs = _functors(f.graph)
    assert [n.i("is_parallel_map") for n in fs] == [0, 1]
    assert [n.i("compact_rows") for n in fs] == [0, 1]
    assert "aten::softmax" in _kinds(fs[0].g("Subgraph"))
    f = _built("c3", args)
    fs = _functors(f.graph)
    assert len(fs) == 1 and "aten::size" not in _kinds(f.graph)
    n = fs[0]
    assert n.i("is_parallel_map") == 1 and n.i("compact_rows") == 1 and n.i("parallel_degree") == 6
    assert list(getattr(n, "is")("is_parallel_args")) == [0, 0, 0]
    kinds = _kinds(n.g("Subgraph"))
    assert "aten::softmax" in kinds and "immut::select" in kinds and kinds[-1] == "aten::gt"


def test_nothing_is_sunk_while_the_head_kernels_are_switched_off():
    from functs_amd._lib import lib
    args = oc.c3_inputs(0, 60, 7)
    lib.fx_set_head_kernel(0)
    try:
        f = _built("c3", args)
    finally:
        lib.fx_set_head_kernel(1)
    assert [n.i("is_parallel_map") for n in _functors(f.graph)] == [0, 1]


def test_a_producer_with_other_readers_is_not_sunk():
    def g(loc: torch.Tensor, conf: torch.Tensor, priors: torch.Tensor):
        l0 = loc[0]
        cxcy = priors[:, :2] + l0[:, :2] * 0.1 * priors[:, 2:]
        wh = priors[:, 2:] * torch.exp(l0[:, 2:] * 0.2)
        boxes = torch.cat([cxcy - wh / 2, cxcy + wh / 2], 1)
        scores = conf[0].softmax(-1)
        out_b: List[torch.Tensor] = []
        out_s: List[torch.Tensor] = []
        for c in range(1, scores.size(1)):
            sc = scores[:, c]
            m = sc > 0.05
            out_b.append(boxes[m])
            out_s.append(sc[m])
        return out_b, out_s, boxes      # the decoded boxes are a result of their own

    def other_decode(loc: torch.Tensor, conf: torch.Tensor, priors: torch.Tensor):
        # the producer only feeds the map, but the merged region is neither one the library has a
        # hand-written kernel for (boxes by cat) nor a row stream (the softmax is a reduction):
        # lowered generically every class would redo the softmax
        l0 = loc[0]
        cxcy = priors[:, :2] + l0[:, :2] * 0.1 * priors[:, 2:]
        wh = priors[:, 2:] * torch.exp(l0[:, 2:] * 0.2)
        boxes = torch.cat([cxcy - wh / 2, cxcy + wh / 2], 1)
        scores = conf[0].softmax(-1)
        out_b: List[torch.Tensor] = []
        out_s: List[torch.Tensor] = []
        for c in range(1, scores.size(1)):
            sc = scores[:, c]
            m = sc > 0.05
            out_b.append(boxes[m])
            out_s.append(sc[m])
        return out_b, out_s

    args = oc.c3_inputs(0, 60, 7)
    for fn in (g, other_decode):
        built = fj.build(fj.script(fn), list(args))
        assert [n.i("is_parallel_map") for n in _functors(built.graph)] == [0, 1], fn.__name__


def test_an_elementwise_producer_sinks_into_a_map_that_streams_rows():
    """No reduction in the merged region: every class evaluates the producer for its own kept rows
    only, nothing is done twice, and the map is a row compaction with a row-stream form."""
    def sigmoid_scores(loc: torch.Tensor, conf: torch.Tensor, priors: torch.Tensor):
        l0 = loc[0]
        cxcy = priors[:, :2] + l0[:, :2] * 0.1 * priors[:, 2:]
        wh = priors[:, 2:] * torch.exp(l0[:, 2:] * 0.2)
        boxes = torch.cat([cxcy - wh / 2, cxcy + wh / 2], 1)
        scores = conf[0].sigmoid()
        out_b: List[torch.Tensor] = []
        out_s: List[torch.Tensor] = []
        for c in range(1, scores.size(1)):
            sc = scores[:, c]
            m = sc > 0.05
            out_b.append(boxes[m])
            out_s.append(sc[m])
        return out_b, out_s

    args = oc.c3_inputs(0, 60, 7)
    built = fj.build(fj.script(sigmoid_scores), list(args))
    assert [n.i("is_parallel_map") for n in _functors(built.graph)] == [1]


def _mixed_body(x: torch.Tensor):
    out = []
    for i in range(x.size(0)):
        r = x[i] * 2 + 1
        out.append(torch.nonzero(r > 1.5).float().sigmoid().exp())
    return out


def test_map_is_split_around_unfusable_nodes():
    """SplitParallelMaps (fait/passes/parallelize_loops.cpp:152-293): each fused stretch of the
    loop body becomes one launch over all iterations; nonzero stays in a loop between them and
    its ragged results travel as a list."""
    f = fj.build(fj.script(_mixed_body), [torch.rand(3, 8)])
    kinds = _kinds(f.graph)
    assert "prim::ParallelMap" not in kinds and "prim::FusionGroup" not in kinds
    assert kinds.count("tssa::ParallelFunctor") == 2 and kinds.count("prim::Loop") == 1
    loop = [n for n in f.graph.nodes() if n.kind() == "prim::Loop"][0]
    body = [n.kind() for n in loop.blocks().__next__().nodes()]
    assert "aten::nonzero" in body and "tssa::ParallelFunctor" not in body
    for fn in _functors(f.graph):
        assert fn.i("is_parallel_map") == 1
    _C._jit_pass_validate(f.graph)


def test_map_without_fusable_work_stays_a_loop():
    def prog(x: torch.Tensor):
        out = []
        for i in range(x.size(0)):
            out.append(torch.nonzero(x[i]))
        return out

    f = fj.build(fj.script(prog), [torch.rand(3, 8)])
    kinds = _kinds(f.graph)
    assert "prim::ParallelMap" not in kinds and "tssa::ParallelFunctor" not in kinds
    assert "prim::Loop" in kinds and "aten::nonzero" in kinds


@pytest.mark.gpu
def test_split_map_runs_on_gpu():
    x = torch.rand(5, 33, generator=torch.Generator().manual_seed(3))
    want = torch.jit.script(_mixed_body)(x)
    f = fj.build(fj.script(_mixed_body), [x])
    got = f(x.cuda())
    assert len(got) == len(want)
    for g, w in zip(got, want):
        assert g.shape == w.shape
        torch.testing.assert_close(g.cpu(), w, rtol=1e-5, atol=1e-6)


def _dependent_loop(x: torch.Tensor, y: torch.Tensor):
    for i in range(3):
        x = x + y[i]      # one working operator: the body alone is not worth a region
    return x


def test_short_dependent_loop_is_unrolled_and_fused():
    """UnrollLoopsWithDeps (fait/passes/unroll_loops.cpp:11-77): a constant-trip loop with a
    carried value whose body did not fuse is written out; the second FuseOps makes one region
    of the three iterations."""
    f = fj.build(fj.script(_dependent_loop), [torch.rand(8), torch.rand(3, 8)])
    kinds = _kinds(f.graph)
    assert "prim::Loop" not in kinds and kinds.count("tssa::ParallelFunctor") == 1
    sub = _functors(f.graph)[0].g("Subgraph")
    assert [n.kind() for n in sub.nodes()].count("aten::add") == 3


def test_long_or_dynamic_loops_are_not_unrolled():
    def prog(x: torch.Tensor, y: torch.Tensor, n: int):
        for i in range(n):
            x = x * 0.5 + y[i]
        return x

    g = fj.script(prog).graph.copy()
    assert not _C._jit_pass_unroll_loops_with_deps(g)
    assert "prim::Loop" in _kinds(g)


def test_unroll_simple_maps():
    """UnrollSimpleMaps (fait/passes/parallelize_loops.cpp:372-456): a constant-trip map that
    only computes from its index and constants is written out."""
    def prog(x: torch.Tensor):
        out = []
        for i in range(3):
            out.append(torch.ones(4) * float(i) + 1.0)
        return out

    g = fj.script(prog).graph.copy()
    _C._jit_pass_parallelize_loops(g)
    assert "prim::ParallelMap" in _kinds(g)
    assert _C._jit_pass_unroll_simple_maps(g)
    kinds = _kinds(g)
    assert "prim::ParallelMap" not in kinds and kinds.count("aten::mul") == 3
    _C._jit_pass_validate(g)
    got = _C._create_function_from_graph("unrolled", g)(torch.zeros(1))
    assert [t.tolist() for t in got] == [[1.0] * 4, [2.0] * 4, [3.0] * 4]


@pytest.mark.gpu
def test_unrolled_loop_runs_on_gpu():
    gen = torch.Generator().manual_seed(5)
    x, y = torch.rand(257, generator=gen), torch.rand(3, 257, generator=gen)
    want = _dependent_loop(x.clone(), y)
    f = fj.build(fj.script(_dependent_loop), [x, y])
    torch.testing.assert_close(f(x.cuda(), y.cuda()).cpu(), want, rtol=1e-6, atol=0)


def test_single_elementwise_op_is_left_to_aten():
    def prog(x: torch.Tensor):
        return x.sigmoid()

    f = fj.build(fj.script(prog), [torch.rand(3, 8)])
    assert not _functors(f.graph)
    assert torch.equal(f(torch.ones(2, 2)), torch.ones(2, 2).sigmoid())


def test_functor_refuses_cpu_tensors():
    f = _built("c1", oc.c1_inputs(0, 64))
    with pytest.raises(RuntimeError, match="GPU only"):
        f(*oc.c1_inputs(0, 64))


def test_validate_rejects_use_before_definition():
    g = torch._C.parse_ir("""
graph(%a : Tensor):
  %one : int = prim::Constant[value=1]()
  %c : Tensor = aten::add(%a, %a, %one)
  %b : Tensor = aten::mul(%c, %a)
  return (%b)""")
    _C._jit_pass_validate(g)
    nodes = [n for n in g.nodes() if n.kind() in ("aten::add", "aten::mul")]
    nodes[1].moveBefore(nodes[0])
    with pytest.raises(RuntimeError, match="before it is defined"):
        _C._jit_pass_validate(g)


# --------------------------------------------------------------------------- gpu
def _cuda(args):
    return [a.cuda() if isinstance(a, torch.Tensor) else a for a in args]


def _cpu(x):
    if isinstance(x, (list, tuple)):
        return [_cpu(t) for t in x]
    return x.cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("size", [64, 1024])
def test_c1_torchscript_gpu(size):
    args = oc.c1_inputs(0, size)
    ref = oc.run("c1", *args)
    got = _built("c1", args)(*_cuda(args))
    assert_exact(got.cpu(), ref, "c1")


@pytest.mark.gpu
@pytest.mark.parametrize("grids", [SMALL_GRIDS, oc.YOLO_GRIDS])
def test_c2_torchscript_gpu(grids):
    args = oc.c2_inputs(0, grids)
    assert oc.threshold_margin(torch.sigmoid(args[0][..., 4]), 0.3) > 1e-6
    rb, rc, ro = oc.run("c2", *args)
    f = _built("c2", args)
    for _ in range(2):  # the second call reuses the compiled variant
        gb, gc, go = _cpu(f(*_cuda(args)))
        assert_boxes_close(gb, rb, "c2 boxes")
        assert_close(gc, rc, "c2 cls")
        assert_close(go, ro, "c2 obj")


@pytest.mark.gpu
@pytest.mark.parametrize("grids,batch", [(SMALL_GRIDS, 3), (oc.YOLO_GRIDS, 16)])
def test_c5_torchscript_gpu(grids, batch):
    args = oc.c5_inputs(0, grids, batch)
    rb, rc, ro = oc.run("c5", *args)
    gb, gc, go = _cpu(_built("c5", args)(*_cuda(args)))
    assert_boxes_close(gb, list(rb), "c5 boxes")
    assert_close(gc, list(rc), "c5 cls")
    assert_close(go, list(ro), "c5 obj")


@pytest.mark.gpu
def test_c5_torchscript_gpu_more_images_than_the_argument_block_has_pointers_for():
    """130 images x 3 results = 390 per-task buffers: the pointer table is uploaded ahead of the
    kernel (the build of the generated row-stream kernel that reads its tables from device memory:
    still one launch), and the results are those of the oracle."""
    import functs_amd.aot as aot
    args = oc.c5_inputs(2, SMALL_GRIDS, 130)
    rb, rc, ro = oc.run("c5", *args)
    f = _built("c5", args)
    print("c5 with 130 images", flush=True)
    for _ in range(2):   # (the second call reuses the borrowed scratch with its table)
        l0, _s = aot.launch_stats()
        gb, gc, go = _cpu(f(*_cuda(args)))
        assert aot.launch_stats()[0] - l0 == 1
        assert len(gb) == 130
        assert_boxes_close(gb, list(rb), "c5 boxes")
        assert_close(gc, list(rc), "c5 cls")
        assert_close(go, list(ro), "c5 obj")


@pytest.mark.gpu
def test_c5_torchscript_gpu_new_batch_size_same_function():
    """parallel_degree is taken from the trip count at run time."""
    args3 = oc.c5_inputs(0, SMALL_GRIDS, 3)
    f = _built("c5", args3)
    for batch in (3, 5, 1):
        args = oc.c5_inputs(batch, SMALL_GRIDS, batch)
        rb, rc, ro = oc.run("c5", *args)
        gb, gc, go = _cpu(f(*_cuda(args)))
        assert_boxes_close(gb, list(rb), "c5 boxes b=%d" % batch)
        assert_close(go, list(ro), "c5 obj b=%d" % batch)


@pytest.mark.gpu
@pytest.mark.parametrize("n_priors,n_cls", [(60, 7), (8732, 81), (33, 2), (1917, 91), (8732, 21), (24564, 21)])
def test_c3_torchscript_gpu(n_priors, n_cls):
    args = oc.c3_inputs(0, n_priors, n_cls)
    rb, rs = oc.run("c3", *args)
    one = _built("c3", args)
    assert len(_functors(one.graph)) == 1
    gb, gs = _cpu(one(*_cuda(args)))
    assert_close(gb, list(rb), "c3 boxes", rtol=1e-5, atol=1e-6)
    assert_close(gs, list(rs), "c3 scores")
    # the two functors of the reference's pipeline give the same bits
    _C._set_sink_producers(False)
    try:
        two = _built("c3", args)
    finally:
        _C._set_sink_producers(True)
    assert len(_functors(two.graph)) == 2
    tb, ts = _cpu(two(*_cuda(args)))
    assert_exact(gb, tb, "c3 boxes, one functor vs two")
    assert_exact(gs, ts, "c3 scores, one functor vs two")


@pytest.mark.gpu
def test_c3_torchscript_gpu_other_numbers_of_priors_same_function():
    """The merged functor is built for the example's shapes; another number of priors gets a
    plan of its own at run time (the class count is part of the function: its trip count)."""
    f = _built("c3", oc.c3_inputs(0, 500, 21))
    assert len(_functors(f.graph)) == 1
    for n in (500, 77, 3000):
        args = oc.c3_inputs(n, n, 21)
        rb, rs = oc.run("c3", *args)
        gb, gs = _cpu(f(*_cuda(args)))
        assert_close(gb, list(rb), "c3 boxes n=%d" % n, rtol=1e-5, atol=1e-6)
        assert_close(gs, list(rs), "c3 scores n=%d" % n)


def test_c4_lstm_is_functionalized_and_keeps_its_loops():
    """Loops with carried state stay host loops; the cell's gate arithmetic and
    both state writes form one region per (step, layer)."""
    args = oc.c4_inputs(0, 5, 16, 2, 1)
    f = fj.script(oc.c4_fn)
    kinds = _kinds(f.graph)
    assert "aten::copy_" not in kinds and kinds.count("immut::select_rev") == 3
    got = f(*args)  # functionalized graph, stock interpreter, CPU
    ref = oc.run("c4", *args)
    for g_, r in zip(got, ref):
        assert torch.equal(g_, r)
    built = fj.build(f, list(args))
    kinds = _kinds(built.graph)
    assert kinds.count("prim::Loop") == 2 and kinds.count("aten::matmul") == 2
    inner = [n for n in _functors(built.graph) if "aten::tanh" in _kinds(n.g("Subgraph"))]
    assert len(inner) == 1
    sub = _kinds(inner[0].g("Subgraph"))
    assert sub.count("immut::select_rev") == 2 and sub.count("aten::sigmoid") == 3


@pytest.mark.gpu
@pytest.mark.parametrize("seq_len,hidden", [(5, 16), (64, 512)])
def test_c4_lstm_torchscript_gpu(seq_len, hidden):
    args = oc.c4_inputs(0, seq_len, hidden, 2, 1)
    ref = oc.run("c4", *args)
    # the product's own program text: it creates its state on x.device (the oracle's text creates
    # it on the default device, which is the host: fills over static shapes run where they say)
    from functs_amd.benchmark import PROGRAMS
    got = fj.build(fj.script(PROGRAMS["c4"]), list(args))(*_cuda(args))
    # 1e-5 per step compounds over the recurrence: 1e-4 at the last step (matmul runs in rocBLAS)
    for name, g_, r in zip(("out", "state_h", "state_c"), got, ref):
        assert_close(g_.cpu(), r, "c4 " + name, rtol=1e-4, atol=1e-6)


@pytest.mark.gpu
def test_c4_lstm_as_hip_graph():
    """Every replay is checked against the eager call, with other work and
    synchronisations of the program in between, and with fresh input values."""
    from functs_amd.benchmark import PROGRAMS
    args0 = oc.c4_inputs(0, 12, 64, 2, 1)
    f = fj.script(PROGRAMS["c4"])
    eager = fj.build(f, list(args0))
    graphed = fj.build(f, list(args0), hip_graph=True)
    for seed in (0, 1, 2, 1):
        args = _cuda(oc.c4_inputs(seed, 12, 64, 2, 1))
        want = eager(*args)
        torch.cuda.synchronize()
        got = graphed(*args)
        junk = torch.rand(4096, device="cuda").sum().item()  # unrelated work between replays
        assert junk > 0
        for g_, w in zip(got, want):
            assert torch.equal(g_, w)
    ref = oc.run("c4", *oc.c4_inputs(1, 12, 64, 2, 1))
    for g_, r in zip(got, ref):
        assert_close(g_.cpu(), r, "graphed c4", rtol=1e-4, atol=1e-6)


@pytest.mark.gpu
def test_every_captured_lstm_clears_a_workspace_of_its_own():
    """Two graphs of one function, of which only the second is replayed, in memory that held other values."""
    from functs_amd.benchmark import PROGRAMS
    args = _cuda(oc.c4_inputs(3, 12, 64, 2, 1))
    f = fj.build(fj.script(PROGRAMS["c4"]), list(oc.c4_inputs(3, 12, 64, 2, 1)))
    want = f(*args)
    torch.cuda.synchronize()
    pool, g0 = torch.cuda.graph_pool_handle(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(g0, pool=pool):
        junk = [torch.full((8192,), 255, dtype=torch.uint8, device="cuda") for _ in range(600)]
    g0.replay()
    torch.cuda.synchronize()
    del junk
    graphs, outs = [torch.cuda.CUDAGraph() for _ in range(2)], []
    for g in graphs:
        with torch.cuda.graph(g, pool=pool):
            outs.append(f(*args))
    for _ in range(3):
        graphs[1].replay()
        torch.cuda.synchronize()
        for got, w in zip(outs[1], want):
            assert torch.equal(got, w)


def test_hip_graph_refuses_row_compaction():
    args = oc.c2_inputs(0, SMALL_GRIDS)
    with pytest.raises(ValueError, match="row-compacting"):
        fj.build(fj.script(oc.c2_fn), list(args), hip_graph=True)


@pytest.mark.gpu
def test_back_to_back_calls_with_changing_inputs():
    """The operator returns when the kept-row counts are known, before its kernels end, so
    consecutive calls overlap on the stream and reuse scratch and the pinned count buffer.
    Alternating inputs with different kept rows must never show a stale size or stale rows."""
    import functs_amd.jit as fj
    from functs_amd.benchmark import PROGRAMS
    from functs_amd.benchmark.inputs import INPUTS
    dev = torch.device("cuda:0")
    a = INPUTS["c5"](0)
    b = INPUTS["c5"](1)
    fn = fj.build(fj.script(PROGRAMS["c5"]), list(a))
    ga = [t.to(dev) for t in a]
    gb = [t.to(dev) for t in b]
    want = {}
    for key, args in (("a", ga), ("b", gb)):
        out = fn(*args)
        torch.cuda.synchronize()
        want[key] = [[t.clone() for t in lst] for lst in out]
    assert [t.shape for t in want["a"][0]] != [t.shape for t in want["b"][0]]
    pending = []
    for it in range(120):
        key, args = (("a", ga), ("b", gb))[it % 2]
        pending.append((key, fn(*args)))          # no synchronisation between calls
    torch.cuda.synchronize()
    for key, out in pending:
        for lst, ref in zip(out, want[key]):
            assert len(lst) == len(ref)
            for t, r in zip(lst, ref):
                assert t.shape == r.shape and torch.equal(t, r)
