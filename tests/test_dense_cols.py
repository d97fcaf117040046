"""An output of rows of four elements whose columns are programs of their own, side by side in one kernel (fx_dense_cols): the
same bits as column by column (fx_region_dense in boxes, the kernel with the short arguments switched off)."""
import pytest
import torch

import functs_amd.jit as fj
from functs_amd import _C, _lib
from functs_amd.benchmark import PROGRAMS


# rows on either side of a wave and a workgroup, one class (another program), rows whose classes end inside a wave, more
# rows than the launch has threads
@pytest.mark.gpu
@pytest.mark.parametrize("n,classes", [(2, 1), (63, 1), (65, 1), (257, 1), (2, 3), (21, 3), (85, 3), (86, 3), (129, 2), (37, 7), (333, 21), (9000, 100)])
def test_side_by_side_and_column_by_column(n, classes):
    g = torch.Generator(device="cuda").manual_seed(n * 101 + classes)
    rois = torch.rand(n, 4, generator=g, device="cuda") * 150
    rois[:, 2:] += rois[:, :2]
    deltas = torch.randn(n, 4 * classes, generator=g, device="cuda")
    deltas.view(-1)[::13] *= 40.0                      # beyond the clamp
    for k, x in enumerate((float("nan"), float("inf"), -float("inf"), -0.0)):
        deltas.view(-1)[k + 4::57] = x
    fn = fj.build(fj.script(PROGRAMS["delta2bbox"]), [rois, deltas])
    assert "lean dense kernel" in " ".join(_C._plan_functors(fn.graph))
    odd = torch.empty(n * 4 * classes + 1, device="cuda")[1:].view(n, 4 * classes).copy_(deltas)   # (not 16-byte aligned)
    print("cols", n, classes, flush=True)
    got = [fn(rois, deltas), fn(rois, odd)]
    _lib.lib.fx_set_dense_lean(0)
    try:
        ref = fn(rois, deltas)
    finally:
        _lib.lib.fx_set_dense_lean(1)
    want = PROGRAMS["delta2bbox"](rois.cpu(), deltas.cpu())
    for t in got:
        assert torch.equal(t.view(torch.int32), ref.view(torch.int32))
        torch.testing.assert_close(t.cpu(), want, rtol=1e-5, atol=1e-3, equal_nan=True)
