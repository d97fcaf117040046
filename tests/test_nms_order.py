"""The finishing workgroup of fx_sort_nms: candidates ordered by buckets of their scores (up to 2 048), by the sort beyond that and
where a bucket holds many; overlaps decided by comparisons, by the product, by the division.  Kept boxes are the oracle's."""
import pytest
import torch

from oracle import nms as onms

import functs_amd._C  # noqa: F401


def _case(n, rows, kind, seed):
    g = torch.Generator().manual_seed(seed)
    xy = torch.rand(rows, 2, generator=g) * 300.0 - 40.0
    wh = torch.rand(rows, 2, generator=g) * 60.0
    if kind == "flat":
        wh[::3, 0] = 0.0                       # boxes of no area
    if kind == "swapped":
        wh[::5] *= -1.0
    boxes = torch.cat([xy, xy + wh], 1)
    scores = torch.zeros(rows, 2)
    at = torch.randperm(rows * 2, generator=g)[:n]
    u = torch.rand(n, generator=g)
    if kind == "equal":
        u = torch.full((n,), 0.5)              # one bucket
    if kind == "steps":
        u = (u * 20).floor() / 20              # twenty of them
    if kind == "far":
        u = u * 0.01
        u[:3] = torch.tensor([1.0, 1.0, 3e30])   # one score far from the others
    scores.view(-1)[at] = 0.06 + 0.9 * u
    return boxes, scores, torch.rand(rows, generator=g) if kind != "equal" else torch.ones(rows)


# few rows: one workgroup an image, nothing handed over; many: several
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1200, 20000])
@pytest.mark.parametrize("n,kind", [(0, "plain"), (1, "plain"), (48, "equal"), (49, "equal"), (700, "plain"), (700, "equal"), (1025, "steps"), (900, "far"),
                                    (2047, "plain"), (2048, "plain"), (2049, "plain"), (600, "flat"), (600, "swapped")])
def test_kept_boxes_are_the_oracles(rows, n, kind):
    boxes, scores, factors = _case(n, rows, kind, n + rows)
    print("order", rows, n, kind, flush=True)
    for thr, max_num in ((0.45, 100), (0.0, 1024), (-0.25, 60)):
        dets, labels = torch.ops.functs.multiclass_nms(boxes.cuda(), scores.cuda(), factors.cuda(), 0.05, thr, max_num, False)
        rd, rl, _ = onms.multiclass_nms(boxes, scores, factors, 0.05, thr, max_num)
        assert torch.equal(labels.cpu(), rl) and torch.equal(dets.cpu(), rd), (thr, max_num)
