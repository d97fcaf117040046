"""The detection head of any number of classes in one launch: rows of class scores that are no whole groups of
four leave fx_head_stream as one run of 16-byte lines per sub-tile.  Bit for bit what the two passes give."""
import pytest
import torch

from functs_amd import configs
from functs_amd._lib import lib
from tests.test_head_stream import _folded, _head, _head_folded, _info, _inputs
from tests.util import assert_exact, run_region


def test_any_number_of_classes_is_one_launch_while_row_stream_kernels_are_on():
    for classes in (1, 2, 3, 5, 13, 81, 91):
        for batch in (None, 3):
            info, p = _info(_head(batch=batch), *_inputs(50, classes, batch or 1))
            assert info[1] == 1 and info[4] == classes and lib.fx_plan_launches(p.handle) == 1
            info, p = _info(_head_folded(batch=batch), *_folded(*_inputs(50, classes, batch or 1)))
            assert info[1] == 1 and lib.fx_plan_launches(p.handle) == 1
    for switch, on in ((lib.fx_set_rowstream, 1), (lib.fx_set_head_kernel, 1), (lib.fx_set_specialization, 1)):
        _, p = _info(_head(), *_inputs(50, 13, 1))
        switch(0)
        try:
            assert lib.fx_plan_launches(p.handle) == 2
        finally:
            switch(on)
    for r in (_head(obj_col=3), _head(half=0.25)):   # another computation
        _, p = _info(r, *_inputs(50, 13, 1))
        assert lib.fx_plan_launches(p.handle) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("n,classes,batch", [(1, 1, None), (5, 1, 2), (64, 2, None), (65, 3, 3), (300, 5, 16), (1000, 6, 1), (777, 7, 5), (22743, 13, 2),
                                             (2000, 81, 3), (901, 91, None), (50, 341, 2)])
def test_bit_exact_against_the_two_passes(n, classes, batch):
    args = _inputs(n, classes, batch or 1, seed=n + classes)
    for r, a in ((_head(batch=batch), args), (_head_folded(batch=batch), _folded(*args))):
        one = run_region("hip", r, *a)
        lib.fx_set_head_kernel(0)
        try:
            two = run_region("hip", r, *a)
        finally:
            lib.fx_set_head_kernel(1)
        assert_exact(one, two, "n=%d classes=%d batch=%s" % (n, classes, batch))


@pytest.mark.gpu
def test_nothing_everything_and_nan_rows():
    for value in (-20.0, 20.0, float("nan")):
        pred, anchors, strides = _inputs(700, 13, 4)
        pred[..., 4] = value
        pred[1, 5, 7] = float("inf")
        r = configs.build_c5(4)
        one = run_region("hip", r, pred, anchors, strides)
        lib.fx_set_head_kernel(0)
        try:
            two = run_region("hip", r, pred, anchors, strides)
        finally:
            lib.fx_set_head_kernel(1)
        assert_exact(one, two, "objectness %g" % value)
        assert [t.shape[0] for t in one[2]] == [700 if value > 0 else 0] * 4
