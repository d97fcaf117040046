"""Programs that write to their arguments in place, between reading them: a region reads its operands where the program does, and
what is written through a view reaches the argument.  Results and arguments are eager mode's."""
from typing import List

import pytest
import torch
from torch import Tensor

import functs_amd.jit as fj
from functs_amd import _C


def whole_argument(x: Tensor, m: Tensor):
    y = x + 1.0
    x.zero_()
    z = y * 2.0 + m
    return z


def row(x: Tensor, m: Tensor):
    y = x + 1.0
    x[0] = 3.0
    z = y * 2.0 + m
    return z


def written_ahead(x: Tensor, m: Tensor):
    x[0:2] = m[0:2] * 2.0
    return x * 3.0 + m


def written_in_a_loop(x: Tensor, m: Tensor):
    out: List[Tensor] = []
    for i in range(4):
        y = x * 2.0 + m
        x.add_(1.0)
        out.append(y)
    return torch.stack(out)


def rows_in_a_loop(x: Tensor, m: Tensor):
    for i in range(8):
        x[i] = x[i] * 2.0 + m[i]
    return x + 1.0


def read_again(x: Tensor, m: Tensor):
    a = x * 2.0 + m
    x.mul_(0.5)
    b = x * 2.0 + m
    return a - b


def columns(x: Tensor, m: Tensor):
    x[1:3, 2:5].fill_(7.0)
    m[:, 0] = x[:, 1] + 2.0
    return x * m + 1.0


def loop_behind(x: Tensor, m: Tensor):
    y = x + m
    out: List[Tensor] = []
    x.zero_()
    for i in range(y.size(0)):
        o = y[i] * 2.0
        out.append(o + x[i])
    return out


def view_kept(x: Tensor, m: Tensor):
    v = x[2]
    y = v * 2.0 + 1.0
    v.zero_()
    return y + m[0], x * 1.0 + 0.0


def view_read_behind(x: Tensor, m: Tensor):
    v = x[2]
    y = v * 2.0 + m[0]
    x.zero_()
    return y, v * 2.0 + 1.0


def from_a_copy(x: Tensor, m: Tensor):
    y = x.clone()
    y[0] = 5.0
    x.copy_(y * 2.0)
    return x + y


def two_arguments_in_a_loop(x: Tensor, m: Tensor):
    for i in range(3):
        x[i, :] = m[i, :] + 1.0
        m[i + 1, :] = x[i, :] * 2.0
    return x + m


def other_argument(x: Tensor, m: Tensor):
    y = x * 2.0 + 1.0
    m.zero_()
    return y * 3.0 + m


def joined(x: Tensor, m: Tensor):
    y = torch.cat([x, m]) * 2.0
    x[1, 2:] = 0.0
    return y + 1.0, torch.cat([x, m]) * 2.0 + 1.0


def in_a_branch(x: Tensor, m: Tensor, flag: bool):
    y = x * 2.0
    if flag:
        x.zero_()
    return y + m + 1.0


def rows_by_a_mask(x: Tensor, m: Tensor):
    s = m * 2.0 + 1.0
    keep = s[:, 0] > 1.0
    x.zero_()
    return x[keep], s[keep]


def rows_by_a_mask_written_behind(x: Tensor, m: Tensor):
    s = m * 2.0 + 1.0
    keep = s[:, 0] > 1.0
    y = x[keep]
    x.zero_()
    return y, s[keep]


def classes_behind(x: Tensor, m: Tensor):
    scores = torch.softmax(x * 2.0 + m, dim=-1)
    x.zero_()
    out: List[Tensor] = []
    for c in range(4):
        s = scores[:, c]
        keep = s > 0.05
        out.append(scores[keep, :])
    return out


def decoded_ahead(loc: Tensor, conf: Tensor, priors: Tensor):
    l0 = loc[0]
    cxcy = priors[:, :2] + l0[:, :2] * 0.1 * priors[:, 2:]
    wh = priors[:, 2:] * torch.exp(l0[:, 2:] * 0.2)
    boxes = torch.zeros_like(priors)
    boxes[:, :2] = cxcy - wh / 2
    boxes[:, 2:] = cxcy + wh / 2
    scores = conf[0].softmax(-1)
    conf.zero_()
    out_b: List[Tensor] = []
    out_s: List[Tensor] = []
    for c in range(1, scores.size(1)):
        sc = scores[:, c]
        m = sc > 0.05
        out_b.append(boxes[m])
        out_s.append(sc[m])
    return out_b, out_s


def written_at_the_end(loc: Tensor, conf: Tensor, priors: Tensor):
    l0 = loc[0]
    cxcy = priors[:, :2] + l0[:, :2] * 0.1 * priors[:, 2:]
    wh = priors[:, 2:] * torch.exp(l0[:, 2:] * 0.2)
    boxes = torch.zeros_like(priors)
    boxes[:, :2] = cxcy - wh / 2
    boxes[:, 2:] = cxcy + wh / 2
    scores = conf[0].softmax(-1)
    out_b: List[Tensor] = []
    out_s: List[Tensor] = []
    for c in range(1, scores.size(1)):
        sc = scores[:, c]
        m = sc > 0.05
        out_b.append(boxes[m])
        out_s.append(sc[m])
    conf.zero_()
    return out_b, out_s


def _head_arguments():
    g = torch.Generator().manual_seed(5)
    return [0.5 * torch.randn(1, 300, 4, generator=g), torch.randn(1, 300, 21, generator=g), torch.rand(300, 4, generator=g)]


def test_a_producer_sinks_into_its_map_unless_its_arguments_are_written():
    for program, functors in ((written_at_the_end, 1), (decoded_ahead, 2)):
        g = fj.script(program).graph.copy()
        _C._jit_pass_fait_pipeline(g, [fj.extract_type_hint_from_tensor(a) for a in _head_arguments()])
        assert [n.kind() for n in g.nodes()].count("tssa::ParallelFunctor") == functors, program.__name__


@pytest.mark.gpu
@pytest.mark.parametrize("program", [decoded_ahead, written_at_the_end])
def test_what_a_map_reads_is_what_the_program_decoded(program):
    ref_args = _head_arguments()
    ref = program(*ref_args)
    print(program.__name__, flush=True)
    fn, args = fj.build(fj.script(program), [a.cuda() for a in _head_arguments()]), [a.cuda() for a in _head_arguments()]
    got = fn(*args)
    assert sum(t.size(0) for t in ref[0]) > 0
    for a, b in zip(got[0] + got[1] + args, ref[0] + ref[1] + ref_args):
        torch.testing.assert_close(a.cpu(), b, rtol=1e-5, atol=1e-5)   # (a few operations and sums of 21 in 32 bits)


PROGRAMS = (whole_argument, row, written_ahead, written_in_a_loop, rows_in_a_loop, read_again, columns, loop_behind, view_kept, view_read_behind,
            from_a_copy, two_arguments_in_a_loop, other_argument, joined, in_a_branch, rows_by_a_mask, rows_by_a_mask_written_behind, classes_behind)


def _arguments(program):
    g = torch.Generator().manual_seed(3)
    args = [torch.randn(8, 16, generator=g), torch.randn(8, 16, generator=g)]
    return args + [True] if program is in_a_branch else args


def _writes(block):
    return sum((n.kind() == "aten::copy_") + sum(_writes(b) for b in n.blocks()) for n in block.nodes())


@pytest.mark.parametrize("program", PROGRAMS)
def test_no_write_is_lost(program):
    g = fj.script(program).graph.copy()
    before = _writes(g.block())
    _C._jit_pass_fait_pipeline(g, [fj.extract_type_hint_from_tensor(a) for a in _arguments(program)])
    assert _writes(g.block()) == before > 0


def test_rows_selected_ahead_of_a_write_are_compacted():
    for program, folded in ((rows_by_a_mask, False), (rows_by_a_mask_written_behind, True)):
        g = fj.script(program).graph.copy()
        _C._jit_pass_fait_pipeline(g, [fj.extract_type_hint_from_tensor(a) for a in _arguments(program)])
        assert ("compact_rows=1" in str(g)) == folded, program.__name__


@pytest.mark.gpu
@pytest.mark.parametrize("program", PROGRAMS)
def test_results_and_arguments_are_eager_modes(program):
    ref_args = _arguments(program)
    ref = program(*ref_args)
    on_gpu = lambda: [a.cuda() if isinstance(a, Tensor) else a for a in _arguments(program)]
    print(program.__name__, flush=True)
    fn, args = fj.build(fj.script(program), on_gpu()), on_gpu()
    got = fn(*args)
    got, ref = ([t] if isinstance(t, Tensor) else list(t) for t in (got, ref))
    assert len(got) == len(ref)
    for a, b in zip(got + args, ref + ref_args):
        if isinstance(a, Tensor):
            torch.testing.assert_close(a.cpu(), b, rtol=1e-5, atol=1e-5)   # (a few operations in 32 bits)
