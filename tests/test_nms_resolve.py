"""The chunks of fx_nms_pairs resolved side by side: chains of overlaps through chunks, everything dead, everything kept,
and waits that are given up at once.  Results are fx_sort_nms's, which a call with counts takes, bit for bit."""
import pytest
import torch

from functs_amd import detection
from functs_amd._lib import lib


def _same(boxes, scores, labels=None, **kw):
    dev = torch.device("cuda:0")
    b, s = boxes.to(dev), scores.to(dev)
    lab = None if labels is None else labels.to(dev)
    counts = torch.full((b.shape[0],), b.shape[1], dtype=torch.int32, device=dev)
    got = detection.batched_nms_batched(b, s, lab, **kw)
    want = detection.batched_nms_batched(b, s, lab, counts=counts, **kw)
    torch.cuda.synchronize()
    assert torch.equal(got.n, want.n) and torch.equal(got.index, want.index) and torch.equal(got.labels, want.labels)
    assert torch.equal(got.dets.view(torch.int32), want.dets.view(torch.int32))
    return got.n.tolist()


def _chain(n, step):
    x = torch.arange(n, dtype=torch.float32) * step
    return torch.stack([x, torch.zeros(n), x + 10.0, torch.full((n,), 10.0)], 1)[None], torch.linspace(1.0, 0.1, n)[None]


def _crowd(tasks, n, span, seed=0):
    g = torch.Generator().manual_seed(seed)
    a = torch.rand(tasks, n, 2, generator=g) * span
    return torch.cat([a, a + 5 + 40 * torch.rand(tasks, n, 2, generator=g)], -1), torch.rand(tasks, n, generator=g), torch.randint(0, 3, (tasks, n), generator=g)


# the first and last row of a chunk, and the sizes at which a wave holds another word per chunk
@pytest.mark.gpu
@pytest.mark.parametrize("n", [129, 192, 193, 1024, 1025, 1984, 1985, 2944, 2945, 4096])
def test_chains_and_crowds(n):
    print("chain n=%d" % n, flush=True)
    kept = _same(*_chain(n, 4.0), iou_threshold=0.3, max_num=1024)          # each box waits for the one before it
    assert kept == [min(1024, (n + 1) // 2)]
    assert _same(*_chain(n, 0.001), iou_threshold=0.3, max_num=1024) == [1]  # one box over all
    cut = min(1024, (n + 3) // 4)                                            # (as few as it takes; fewer are walked)
    assert _same(*_chain(n, 20.0), iou_threshold=0.3, max_num=cut) == [cut]
    assert _same(*_chain(n, 20.0), iou_threshold=0.3, max_num=cut - 1) == [cut - 1]
    b, s, lab = _crowd(2, n, 300.0)
    _same(b, s, lab, iou_threshold=0.3, max_num=1024)
    _same(b, s, lab, iou_threshold=0.6, max_num=cut)
    _same(b, s, lab, iou_threshold=0.6, max_num=17)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1025, 1985, 2100, 4096])
def test_waits_that_are_given_up(n):
    b, s, lab = _crowd(3, n, 200.0, seed=n)
    s[1, : n - 70] = float("-inf")                                           # few candidates
    s[2] = float("nan")                                                      # none
    for polls in (0, 1, 3):
        print("n=%d polls=%d" % (n, polls), flush=True)
        lib.fx_set_stream_spin_limit(polls)
        try:
            kept = _same(b, s, lab, iou_threshold=0.4, max_num=1024)
        finally:
            lib.fx_set_stream_spin_limit(4000)
        assert kept == _same(b, s, lab, iou_threshold=0.4, max_num=1024) and kept[2] == 0


# both third launches, and rows of which fewer are kept than the outputs hold
@pytest.mark.gpu
@pytest.mark.parametrize("n,max_num", [(129, 1024), (1024, 1024), (1025, 1024), (1025, 256), (4096, 1023)])
def test_rows_past_the_kept_ones_are_zero_whatever_the_outputs_held(n, max_num):
    import ctypes
    from functs_amd._lib import FxNmsDesc, check
    b, s, lab = (t.cuda() for t in _crowd(2, n, 60.0, seed=n))
    print("n=%d max_num=%d" % (n, max_num), flush=True)
    results = []
    for fn, ws in ((lib.fx_nms_pairs, torch.empty(lib.fx_nms_pairs_workspace_bytes(2, n), dtype=torch.uint8, device="cuda")),
                   (lib.fx_sort_nms, torch.zeros(lib.fx_sort_nms_workspace_bytes(2, 4096), dtype=torch.uint8, device="cuda"))):
        out = (torch.full((2, max_num, 5), float("nan"), device="cuda"), torch.full((2, max_num), -7, dtype=torch.long, device="cuda"),
               torch.full((2, max_num), -7, dtype=torch.long, device="cuda"), torch.full((2,), -7, dtype=torch.int32, device="cuda"))
        d = FxNmsDesc()
        d.n_tasks, d.rows, d.max_num, d.key_capacity, d.score_thr, d.iou_thr = 2, n, max_num, 4096, float("-inf"), 0.3
        d.boxes, d.boxes_task_stride, d.scores, d.scores_task_stride = b.data_ptr(), b.stride(0), s.data_ptr(), s.stride(0)
        d.labels, d.labels_task_stride = lab.data_ptr(), lab.stride(0)
        d.dets, d.out_labels, d.out_index, d.n_out = (t.data_ptr() for t in out)
        d.workspace, d.workspace_bytes = ws.data_ptr(), ws.numel()
        check(fn(ctypes.byref(d), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        results.append(out)
    (dets, labels, index, kept), want = results
    assert all(torch.equal(a, w) for a, w in zip(results[0], want))
    for t in range(2):
        k = int(kept[t])
        assert 0 < k < max_num and not bool(dets[t, k:].any()) and not bool(labels[t, k:].any()) and not bool(index[t, k:].any())
