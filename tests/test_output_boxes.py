"""Outputs computed in boxes of their elements (fx_lower.cpp, Lowerer::boxesOf): one program per box,
cut where the range tests of cat / stack / in-place slices change their answer.  Values against
stock PyTorch at extents around lane groups and work items, for the emulator and the GPU."""
import os
import re

import pytest
import torch

from functs_amd import Region
from tests.util import assert_close, assert_exact, run_region

# a corner is the difference of a centre and half a size of at most e^4 / 2 = 27.3, whose exponentials
# differ by a few units in the last place: four of them (2^-23 * 27.3 each) whatever the difference is
CANCELLED = 4 * 27.3 * 2.0 ** -23
BACKENDS = ["emul", pytest.param("hip", marks=pytest.mark.gpu)]


def corners(x, a):
    """x [n, 4], a [m, 4]: a cat over rows of two corner decodes, then in-place edits of columns."""
    def decode(t, scale):
        xy, wh = t[:, :2] * scale, t[:, 2:].clamp(-4.0, 4.0).exp() * 0.5
        return torch.cat([xy - wh, xy + wh], 1)
    r = torch.cat([decode(x, 0.1), decode(a, 0.2)], 0)
    r[:, 0::2] = r[:, 0::2].clamp(0.0, 9.0)
    r[:, 3] = r[:, 1] + 1.0
    return r


def corners_region(n, m, per_task=0):
    r = Region(max(per_task, 1), per_task > 0)
    x, a = r.tensor_input(rank=2, per_task=per_task > 0), r.tensor_input(rank=2)

    def decode(t, scale):
        xy, wh = t.slice(1, 0, 2) * scale, t.slice(1, 2, 4).clamp(-4.0, 4.0).exp() * 0.5
        return r.cat([xy - wh, xy + wh], 1)
    v = r.cat([decode(x, 0.1), decode(a, 0.2)], 0)
    v = v.slice_rev(v.slice(1, 0, 4, 2).clamp(0.0, 9.0), 1, 0, 4, 2)
    v = v.select_rev(v.select(1, 1) + 1.0, 1, 3)
    r.output(v)
    r.finalize()
    return r


def n_programs(region, *args):
    return int(re.search(r"n_entries = (\d+)", region.spec_source(*args)).group(1))


@pytest.mark.parametrize("backend", BACKENDS)
@pytest.mark.parametrize("n,m", [(1, 1), (3, 5), (64, 1), (63, 193), (257, 300), (1025, 2)])
def test_rows_and_columns(backend, n, m):
    g = torch.Generator().manual_seed(n)
    x, a = torch.randn(n, 4, generator=g) * 30, torch.randn(4, m, generator=g).t()   # (a: strides 1, m)
    r = corners_region(n, m)
    (got,) = run_region(backend, r, x, a)
    assert_close(got, corners(x, a), atol=CANCELLED)
    assert n_programs(r, x, a) == 8   # two parts of four columns


@pytest.mark.parametrize("backend", BACKENDS)
def test_tasks_of_a_map(backend):
    g = torch.Generator().manual_seed(7)
    xs, a = [torch.randn(n, 4, generator=g) for n in (65, 65, 30)], torch.randn(9, 4, generator=g)   # two task classes
    r = corners_region(65, 9, per_task=3)
    (got,) = run_region(backend, r, xs, a)
    for o, x in zip(got, xs):
        assert_close(o, corners(x, a), atol=CANCELLED)


@pytest.mark.parametrize("backend", BACKENDS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16, torch.int32, torch.int64])
@pytest.mark.parametrize("dims", [(5, 7), (2, 3, 131)])
def test_types_and_whole_groups(backend, dtype, dims):
    """Many narrow parts along the last dimension, odd widths: boxes that end inside a lane group."""
    if backend == "emul" and dtype == torch.float16:
        pytest.skip("the emulator has no fp16")
    g = torch.Generator().manual_seed(3)
    parts = [torch.randint(-9, 9, dims[:-1] + (w,), generator=g).to(dtype) for w in (dims[-1], 1, 2, 4, 6)]
    r = Region()
    ins = [r.tensor_input(dtype, len(dims)) for _ in parts]
    last = len(dims) - 1
    r.output(r.cat([(v + 1) * 2 if i % 2 else v * 3 - 1 for i, v in enumerate(ins)] + [v + 5 - 2 for v in ins], last))
    r.finalize()
    ref = torch.cat([(v + 1) * 2 if i % 2 else v * 3 - 1 for i, v in enumerate(parts)] + [v + 5 - 2 for v in parts], last)
    (got,) = run_region(backend, r, *parts)
    assert_exact(got, ref)
    assert (n_programs(r, *parts) > 2) == (dtype != torch.int64)


@pytest.mark.parametrize("backend", BACKENDS)
@pytest.mark.parametrize("w", [8, 33, 200])
def test_a_reduction_inside_a_box(backend, w):
    """A softmax whose rows are one box of the output: its rows are reduced across a wave."""
    g = torch.Generator().manual_seed(w)
    x, y = torch.randn(37, w, generator=g), torch.randn(37, 3, generator=g)
    r = Region()
    a, b = r.tensor_input(rank=2), r.tensor_input(rank=2)
    r.output(r.cat([b * 2.0 + 1.0, b.sigmoid(), a.softmax(1), b.exp() - 1.0, (b + 3.0) * 0.5, b.tanh()], 1))
    r.finalize()
    (got,) = run_region(backend, r, x, y)
    assert_close(got, torch.cat([y * 2 + 1, y.sigmoid(), x.softmax(1), y.exp() - 1, (y + 3) * 0.5, y.tanh()], 1), rtol=2e-6, atol=1e-6)


def test_what_stays_whole():
    # a triangle's test moves with two coordinates, an index's with data: no box answers them
    r = Region()
    a = r.tensor_input(rank=2)
    r.output(r.op("TRIU", a.exp() + a.sigmoid() * 2.0 - 1.0, 0))
    r.finalize()
    assert n_programs(r, torch.randn(9, 9)) == 1
    r = Region()
    a = r.tensor_input(rank=2)
    r.output(r.cat([a, a + 1.0], 0))   # short
    r.finalize()
    assert n_programs(r, torch.randn(9, 9)) == 1


@pytest.mark.parametrize("backend", BACKENDS)
@pytest.mark.parametrize("batch,a,w,hw", [(1, 1, 5, (1, 1)), (2, 3, 7, (5, 3)), (1, 3, 85, (7, 6)), (3, 2, 6, (1, 9))])
def test_divisions_that_come_out_even(backend, batch, a, w, hw):
    """Flattened maps of two levels and repeated rows: the row number is taken apart into the map's
    coordinates (n = (y * w + x) * a + anchor), and the divisions of the views need no code."""
    g = torch.Generator().manual_seed(w)
    maps = [torch.randn(batch, a * w, h, v, generator=g) for h, v in (hw, (2 * hw[0], hw[1] + 1))]
    rois = torch.randn(sum(m.size(2) * m.size(3) for m in maps), 4, generator=g)
    r = Region()
    ins, ri = [r.tensor_input(rank=4) for _ in maps], r.tensor_input(rank=2)
    flat = []
    for v, m in zip(ins, maps):
        flat.append(v.permute(0, 2, 3, 1).view(batch, m.size(2) * m.size(3) * a, w))
    p = r.cat(flat, 1)
    p = p.slice_rev(p.slice(2, 0, 2).sigmoid(), 2, 0, 2)
    rep = ri.repeat(1, a).view(rois.size(0) * a, 4)
    xy, wh = p.slice(2, 0, 2) + rep.slice(1, 0, 2), (rep.slice(1, 2, 4) - rep.slice(1, 0, 2)) * p.slice(2, 2, 4).exp()
    r.output(p)
    r.output(r.cat([xy - wh * 0.5, xy + wh * 0.5], 2))
    r.finalize()

    q = torch.cat([m.permute(0, 2, 3, 1).reshape(batch, -1, w) for m in maps], 1)
    q[..., :2] = q[..., :2].sigmoid()
    ref = rois.repeat(1, a).view(-1, 4)
    rxy, rwh = q[..., :2] + ref[:, :2], (ref[:, 2:] - ref[:, :2]) * q[..., 2:4].exp()
    got = run_region(backend, r, *maps, rois)
    assert_close(got[0], q)
    # sums of two halves that may cancel: a few units in the last place of the larger one
    top = max(1.0, float(rxy.abs().max()), float(rwh.abs().max()))
    assert_close(got[1], torch.cat([rxy - rwh * 0.5, rxy + rwh * 0.5], 2), atol=4 * top * 2.0 ** -23)
    assert n_programs(r, *maps, rois) >= 8
    assert "ITDIV" not in r.disasm(*maps, rois) and "ITMOD" not in r.disasm(*maps, rois)


@pytest.mark.parametrize("backend", BACKENDS)
@pytest.mark.parametrize("c,n", [(8, 8), (9, 64), (10, 33), (23, 70), (64, 260)])
def test_transposed_boxes(backend, c, n):
    """Boxes that turn a matrix over: lane groups along the columns, lanes along the rows, and what is
    left of the last group in a box of its own."""
    g = torch.Generator().manual_seed(c)
    x, y = torch.randn(2, c, n, generator=g), torch.randn(2, 3, n, generator=g)
    r = Region()
    a, b = r.tensor_input(rank=3), r.tensor_input(rank=3)
    parts = [b.sigmoid() * 2.0 - 1.0, a, b.exp() + 1.0, a * 0.5 + 2.0, b.tanh() - 1.0, (b + 1.0) * (b - 1.0)]
    r.output(r.cat([v.transpose(1, 2) for v in parts], 2))
    r.finalize()
    (got,) = run_region(backend, r, x, y)
    ref = torch.cat([y.sigmoid() * 2 - 1, x, y.exp() + 1, x * 0.5 + 2, y.tanh() - 1, (y + 1) * (y - 1)], 1).transpose(1, 2)
    assert_close(got, ref, atol=2.0 ** -22)   # (differences of values near 1)
    assert n_programs(r, x, y) >= 6 + (2 if c % 4 else 0)


def _decode_args():
    from functs_amd.benchmark.inputs import INPUTS
    return INPUTS["c3"](0)


@pytest.mark.parametrize("first", [True, False])
def test_a_plan_does_not_remember_the_switch_it_was_made_under(first):
    """A region whose whole form is linked runs that whenever compiled kernels are on, in boxes while they
    are off, whatever held when it was planned first."""
    from functs_amd import aot, configs
    r, args = configs.build_c3_decode(), _decode_args()
    try:
        seen = {}
        for on in (first, not first, first, not first):
            aot.enable(on)
            seen.setdefault(on, set()).add((r.spec_key(*args), r.specialized(*args), n_programs(r, *args)))
    finally:
        aot.enable(True)
    assert [len(v) for v in seen.values()] == [1, 1]
    (key_on, linked, whole), (key_off, off, boxes) = seen[True].pop(), seen[False].pop()
    assert linked and whole == 2 and not off and boxes > 2 and key_on != key_off


@pytest.mark.gpu
def test_both_forms_of_a_linked_region_on_the_device():
    from functs_amd import aot, configs
    r, args = configs.build_c3_decode(), [t.cuda() for t in _decode_args()]
    outs, ran = [], []
    try:
        for on in (False, True, False):
            aot.enable(on)
            before = aot.launch_stats()
            outs.append([t.clone() for t in r(*args)])
            ran.append(aot.launch_stats()[1] - before[1])
    finally:
        aot.enable(True)
    assert ran == [0, 1, 0]
    for got in outs[1:]:
        for a, b in zip(got, outs[0]):
            assert torch.equal(a, b)


def test_a_capture_leaves_the_whole_form_and_on_request_the_boxes(tmp_path):
    from functs_amd import aot
    x, a = torch.randn(50, 4), torch.randn(20, 4)
    entries = lambda d: sorted(int(re.search(r"n_entries = (\d+)", (d / f).read_text()).group(1)) for f in os.listdir(d))
    with aot.capture(str(tmp_path / "whole")):
        aot._plan_region(corners_region(50, 20), x, a)
    assert entries(tmp_path / "whole") == [1]
    with aot.capture(str(tmp_path / "both"), boxes=True):
        aot._plan_region(corners_region(50, 20), x, a)
    assert entries(tmp_path / "both") == [1, 8] and set(os.listdir(tmp_path / "whole")) < set(os.listdir(tmp_path / "both"))
    # one of the two is compiled: the whole form where it is short enough, else the boxes
    whole = os.listdir(tmp_path / "whole")[0][:-4]
    assert aot._units_to_compile(str(tmp_path / "both"), "dense") == [whole] == aot._units_to_compile(str(tmp_path / "both"), "auto")
    limit, aot.AUTO_TABLE_INSNS = aot.AUTO_TABLE_INSNS, 100
    try:
        (boxes,) = aot._units_to_compile(str(tmp_path / "both"), "auto")
    finally:
        aot.AUTO_TABLE_INSNS = limit
    assert boxes != whole
