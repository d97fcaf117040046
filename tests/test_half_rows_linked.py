"""The loop over rows of 16-bit elements, linked as a compiled kernel: the lean dense kernel's loads of four items
without a branch, groups at the end of a row from the row's last four elements, two roundings an instruction."""
import pytest
import torch

from functs_amd import Region
from functs_amd._lib import lib
from tests.test_half_groups import DTYPES, _same
from tests.util import run_region


def _loop(dtype):
    r = Region()
    b = r.tensor_input(dtype, 2)
    n = r.scalar_input("int")
    i = r.loop_var()
    r.output(r.op("FORALL_SELECT_REV", b, b.select(0, i) + 1, 0, 0, n))
    return r.finalize()


def _data(dtype, rows, cols):
    bits = torch.randint(-(1 << 15), 1 << 15, (rows, cols), generator=torch.Generator().manual_seed(cols)).to(torch.int16)
    return bits.view(dtype)                                      # every pattern: NaN, infinities, subnormals


def test_the_loops_are_linked():
    for dtype in DTYPES:
        for rows, cols in ((3, 5), (1025, 4097), (1400003, 3)):
            r = _loop(dtype)
            arr, n, _ = r._flatten((torch.empty(rows, cols, dtype=dtype), rows))
            assert lib.fx_plan_specialized(r.plan(arr, n).handle) == 1


# 4 M elements and more take four items a wave: rows without a ragged group, with one of each size, of fewer elements than a
# group; fewer elements take one item
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,cols,lo", [(1, 1, 0), (3, 5, 1), (64, 64, 0), (1000, 4000, 0), (1025, 4096, 0), (1025, 4097, 1), (1027, 4098, 3),
                                          (1029, 4099, 5), (5, 1000001, 2), (1400003, 3, 0), (1400003, 3, 1), (1100001, 4, 1), (900001, 5, 0), (700001, 7, 3)])
def test_rows_and_columns(dtype, rows, cols, lo):
    x = _data(dtype, rows, cols + lo).cuda()[:, lo:]
    _same(run_region("hip", _loop(dtype), x, rows)[0], x.cpu() + 1)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
def test_loads_that_are_not_consecutive(dtype):
    x = _data(dtype, 1027, 4099 * 2).cuda()
    for y in (x.t(), x[:, ::2], x.t()[3:, 1:]):
        _same(run_region("hip", _loop(dtype), y, y.shape[0])[0], y.cpu() + 1)
