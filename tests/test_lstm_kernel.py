"""The stacked-LSTM recurrence as one persistent kernel (fx_lstm_stack) against the oracle (stock
TorchScript on the CPU, oracle/configs.py c4_fn, itself pinned against torch.nn.LSTM in
tests/test_oracle.py).  Reference loop: functs/benchmark/ai_model/lstm/lstm.py:79-133.
Tolerance: 1e-4 relative, the bound stated for 64 dependent steps of fp32 arithmetic whose sums
are taken in another order than the oracle's BLAS takes them, plus 5e-6 absolute: a gate is a sum
of up to 2 x 1024 products of magnitude 0.1, whose rounding error (a few 1e-6) does not shrink
with the result when that happens to be near zero.
On the CPU, the kernel's schedule (diagonals t + j, two parities of the h buffer) and its
hand-over protocol (values tagged with their step, bounded polls, the tag base carried from launch
to launch) run with one host thread per workgroup (tests/support/lstm_emul.cpp)."""
import contextlib
import ctypes

import pytest
import torch

from oracle import configs as oc

RTOL = 1e-4
ATOL = 5e-6


def _inputs(seed, T, H, L, B):
    x, wih, whh, bih, bhh = oc.c4_inputs(seed, seq_len=T, hidden=H, layers=L, batch=B)
    g = torch.Generator().manual_seed(seed + 99)
    h0 = torch.rand(L, B, H, generator=g) * 0.2 - 0.1
    c0 = torch.rand(L, B, H, generator=g) * 0.2 - 0.1
    return x, wih, whh, bih, bhh, h0, c0


def _reference(x, wih, whh, bih, bhh, h0, c0):
    """The loop nest of the oracle's c4_fn with initial states (c4_fn starts from zeros)."""
    T, B, H = x.shape
    L = wih.size(0)
    out = torch.zeros(T, B, H)
    sh, sc = h0.clone(), c0.clone()
    for t in range(T):
        cur = x[t]
        for j in range(L):
            ih = torch.matmul(cur, wih[j]) + bih[j]
            hh = torch.matmul(sh[j], whh[j]) + bhh[j]
            i, f = torch.sigmoid(ih[0] + hh[0]), torch.sigmoid(ih[1] + hh[1])
            g, o = torch.tanh(ih[2] + hh[2]), torch.sigmoid(ih[3] + hh[3])
            c2 = f * sc[j] + i * g
            h2 = o * torch.tanh(c2)
            sc[j], sh[j] = c2, h2
            cur = h2
        out[t] = cur
    return out, sh, sc


def _close(got, ref, what):
    for g, r, n in zip(got, ref, ("out", "state_h", "state_c")):
        assert g.shape == r.shape, (what, n)
        err = (g.double() - r.double()).abs()
        bad = err > ATOL + RTOL * r.double().abs()
        assert not bool(bad.any()), "%s %s: %d beyond rtol %g (max err %g)" % (what, n, int(bad.sum()), RTOL, err.max())


def test_reference_with_zero_states_is_the_oracle():
    x, wih, whh, bih, bhh, _, _ = _inputs(0, 7, 32, 2, 1)
    z = torch.zeros(2, 1, 32)
    ref = _reference(x, wih, whh, bih, bhh, z, z)
    orc = oc.run("c4", x, wih, whh, bih, bhh)
    for a, b in zip(ref, orc):
        assert torch.allclose(a, b, rtol=1e-6, atol=1e-7)


def _emul(x, wih, whh, bih, bhh, h0, c0, spin=1 << 30, skip=-1, launches=1, base0=0):
    from tests.support import emul
    so = emul.lstm_emul()
    T, B, H = x.shape
    L = wih.size(0)
    out, sh, sc = torch.zeros(T, B, H), torch.zeros(L, B, H), torch.zeros(L, B, H)
    ts = [None if t is None else t.contiguous() for t in (x, wih, whh, bih, bhh, h0, c0)]
    err = so.fx_lstm_emul(*[None if t is None else t.data_ptr() for t in ts], out.data_ptr(), sh.data_ptr(),
                          sc.data_ptr(), T, B, H, L, spin, skip, launches, base0)
    return (out, sh, sc), err


@pytest.mark.parametrize("T,H,L,B", [(1, 32, 1, 1), (5, 32, 2, 1), (9, 64, 3, 2), (4, 32, 4, 3), (12, 96, 2, 1)])
def test_schedule_and_barrier_on_host_threads(T, H, L, B):
    args = _inputs(T * 7 + L, T, H, L, B)
    got, err = _emul(*args)
    assert err == 0
    _close(got, _reference(*args), "emul T=%d H=%d L=%d B=%d" % (T, H, L, B))


def test_launches_in_a_row_share_a_workspace_cleared_once():
    """The last workgroup to leave moves the tag base past the launch's tags (-1: it did not), so
    the values the next launch finds never carry a tag it waits for - also for the shortest
    sequences, whose tags would repeat from launch to launch otherwise."""
    args = _inputs(11, 6, 64, 3, 2)
    got, err = _emul(*args, launches=3)
    assert err == 0
    _close(got, _reference(*args), "third launch")
    args = _inputs(12, 1, 32, 2, 1)
    got, err = _emul(*args, launches=4)
    assert err == 0
    _close(got, _reference(*args), "fourth launch of a one-step sequence")


def test_the_tag_base_starts_over_before_it_wraps():
    args = _inputs(13, 5, 32, 2, 1)
    got, err = _emul(*args, launches=3, base0=0x80000000 - 8)
    assert err == 0
    _close(got, _reference(*args), "launch after the tags were cleared")


def test_no_initial_state_means_zeros():
    x, wih, whh, bih, bhh, _, _ = _inputs(5, 6, 32, 2, 2)
    got, err = _emul(x, wih, whh, bih, bhh, None, None)
    assert err == 0
    z = torch.zeros(2, 2, 32)
    _close(got, _reference(x, wih, whh, bih, bhh, z, z), "zero state")


def test_a_wait_that_cannot_end_is_given_up():
    """One workgroup stops writing: every other one must give up after the poll limit, set the
    error word and return (on the GPU the kernel then ends instead of hanging)."""
    args = _inputs(3, 6, 32, 2, 1)
    _, err = _emul(*args, spin=2000, skip=5)
    assert err == 1


def test_after_a_given_up_wait_the_workspace_refuses_work_until_it_is_cleared():
    """The launch that gives up fills its results with NaN; the next launch on the same workspace
    (whatever the host did with the error report in between) does no step, reports the error
    again and returns NaN; on a cleared workspace the sequence runs."""
    from tests.support import emul
    so = emul.lstm_emul()
    args = _inputs(4, 6, 32, 2, 1)
    x = args[0]
    T, B, H = x.shape
    L = args[1].size(0)
    out, sh, sc = torch.zeros(T, B, H), torch.zeros(L, B, H), torch.zeros(L, B, H)
    ts = [t.contiguous() for t in args]
    bits = so.fx_lstm_emul_give_up(*[t.data_ptr() for t in ts], out.data_ptr(), sh.data_ptr(), sc.data_ptr(),
                                   T, B, H, L, 2000, 5)
    assert bits & 1, "the first launch did not give up"
    assert bits & 2, "the launch that gave up left values that look like results"
    assert bits & 4 and bits & 8, "the launch on the workspace of a given-up wait ran"
    assert bits & 16, "the launch on the cleared workspace failed"
    _close((out, sh, sc), _reference(*args), "launch on the cleared workspace")


@pytest.mark.parametrize("T,H,L,B,launches", [(1, 32, 1, 2, 5), (1, 32, 4, 2, 3), (2, 32, 2, 2, 4), (7, 32, 3, 3, 3), (6, 64, 2, 2, 2)])
def test_words_are_cleared_two_steps_ahead_on_host_threads(T, H, L, B, launches):
    """The hand-over of the rows kernel: values without tags in four slots, cleared two steps ahead,
    launches in a row (of fewer steps than slots as well) on one workspace that is cleared once."""
    from tests.support import emul
    so = emul.lstm_emul()
    args = _inputs(T * 5 + L, T, H, L, B)
    out, sh, sc = torch.zeros(T, B, H), torch.zeros(L, B, H), torch.zeros(L, B, H)
    ts = [t.contiguous() for t in args]
    err = so.fx_lstm_emul_words(*[t.data_ptr() for t in ts], out.data_ptr(), sh.data_ptr(), sc.data_ptr(), T, B, H, L, 1 << 30, -1, launches)
    assert err == 0
    _close((out, sh, sc), _reference(*args), "words T=%d H=%d L=%d B=%d" % (T, H, L, B))
    if T > 1:   # a workgroup that stops writing: the others give up
        assert so.fx_lstm_emul_words(*[t.data_ptr() for t in ts], out.data_ptr(), sh.data_ptr(), sc.data_ptr(), T, B, H, L, 2000, 5, 1) == 1


@pytest.mark.parametrize("seed", range(12))
def test_launches_that_may_overlap_fit_the_device_together(seed):
    """A workgroup waits for all others of its launch, so launches on several streams may only run at the
    same time when all their workgroups get places: random programs over the grids of the kernel's forms."""
    import ctypes
    from tests.support import emul
    so = emul.lstm_emul()
    device = so.fx_lstm_need_of(256, 1)
    assert device == so.fx_lstm_need_of(512, 2) == so.fx_lstm_need_of(512, 3) and so.fx_lstm_need_of(8, 16) * 512 == device
    forms = [(256, 1), (128, 1), (256, 2), (192, 1), (128, 3), (64, 1), (32, 2), (8, 8)]
    forms = forms[seed % 3:] if seed % 2 else forms[: 3 + seed % 4]
    needs = (ctypes.c_uint32 * len(forms))(*[so.fx_lstm_need_of(*f) for f in forms])
    waits = ctypes.c_int()
    assert so.fx_lstm_groups_emul(seed, 1, 200, needs, len(forms), device, ctypes.byref(waits)) <= device and waits.value == 0   # one stream never waits
    for streams in (2, 3, 7):
        assert so.fx_lstm_groups_emul(seed, streams, 300, needs, len(forms), device, ctypes.byref(waits)) <= device and waits.value > 0
    halves = (ctypes.c_uint32 * 1)(so.fx_lstm_need_of(256, 2))
    assert so.fx_lstm_groups_emul(seed, 2, 100, halves, 1, device, ctypes.byref(waits)) == device and waits.value == 0   # two halves overlap


@pytest.mark.parametrize("waves,registers", [(5, 40), (5, 72), (7, 72), (8, 92), (8, 120), (10, 64), (10, 96), (11, 112), (12, 104), (12, 152)])
def test_workgroups_that_share_a_compute_unit_fit_however_their_waves_are_dealt(waves, registers):
    """The share of a compute unit that a launch is counted with is enough when the odd waves of all
    workgroups go to the same SIMD: (waves, registers) of a workgroup beside every other kind."""
    from tests.support import emul
    so = emul.lstm_emul()
    kinds = [(5, 40), (7, 72), (8, 92), (10, 96), (11, 112), (12, 152)] + [(waves, registers)]
    unit = so.fx_lstm_need_of(1, 1)

    def share(w, v):   # resident workgroups as the runtime counts them: waves of the whole unit
        per_cu = 4 * min(8, 512 // v) // (so.fx_lstm_block_of(64 * w) // 64)
        return so.fx_lstm_need_of(1, per_cu)
    for w, v in kinds:
        for n in range(unit // share(waves, registers) + 1):
            m = (unit - n * share(waves, registers)) // share(w, v)   # the rest of the unit, filled up
            most = [n * -(-waves // 4), m * -(-w // 4)]               # waves on the fullest SIMD
            assert sum(most) <= 8 and most[0] * registers + most[1] * v <= 512, (w, v, n, m)


@contextlib.contextmanager
def lstm_form(form):
    """Launches of this thread take `form` (FX_LSTM_FORM_..., without the prefix), whatever ran before."""
    from functs_amd._lib import C, lib
    before = lib.fx_set_lstm_form(C["FX_LSTM_FORM_" + form])
    try:
        yield
    finally:
        lib.fx_set_lstm_form(before)


def _gpu(x, wih, whh, bih, bhh, h0, c0, launches=1, form="ANY"):
    """`launches` calls in a row on one workspace that is cleared once; the last call's results."""
    with lstm_form(form):
        return _gpu_launches(x, wih, whh, bih, bhh, h0, c0, launches, form)


def _gpu_launches(x, wih, whh, bih, bhh, h0, c0, launches, form):
    from functs_amd._lib import C, check, lib
    dev = torch.device("cuda:0")
    T, B, H = x.shape
    L = wih.size(0)
    ts = [None if t is None else t.contiguous().to(dev) for t in (x, wih, whh, bih, bhh, h0, c0)]
    nbytes = lib.fx_lstm_stack_workspace_bytes(B, H, L)
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    assert ws.data_ptr() % 256 == 0
    stream = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    for _ in range(launches):
        out = torch.full((T, B, H), float("nan"), device=dev)
        sh, sc = torch.full((L, B, H), float("nan"), device=dev), torch.full((L, B, H), float("nan"), device=dev)
        print("fx_lstm_stack T=%d B=%d H=%d L=%d" % (T, B, H, L), flush=True)
        check(lib.fx_lstm_stack(*[None if t is None else t.data_ptr() for t in ts], out.data_ptr(), sh.data_ptr(),
                                sc.data_ptr(), T, B, H, L, ws.data_ptr(), nbytes, stream))
        torch.cuda.synchronize()
        assert lib.fx_async_error(1) == 0
        assert form == "ANY" or lib.fx_lstm_form() == C["FX_LSTM_FORM_" + form]
    return out.cpu(), sh.cpu(), sc.cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,L,B", [(1, 32, 1, 1), (5, 64, 2, 1), (9, 128, 3, 2), (4, 32, 4, 3), (16, 256, 2, 1),
                                     (64, 512, 2, 1), (6, 512, 4, 16), (8, 1024, 1, 2), (7, 1024, 2, 1)])
def test_kernel_against_the_oracle(T, H, L, B):
    """Row by row, the form that serves every size."""
    args = _inputs(T + H + L, T, H, L, B)
    _close(_gpu(*args, form="SINGLE"), _reference(*args), "gpu T=%d H=%d L=%d B=%d" % (T, H, L, B))


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,L,B", [(5, 64, 2, 1), (7, 64, 4, 2), (8, 64, 1, 3), (9, 128, 1, 1), (6, 128, 4, 2), (6, 256, 3, 2), (5, 256, 4, 1),
                                     (7, 512, 1, 1), (70, 512, 3, 1), (4, 512, 4, 2)])
def test_row_by_row_at_the_sizes_that_fit_a_die(T, H, L, B):
    """What captured launches and launches beside others may take there."""
    args = _inputs(T + H + L, T, H, L, B)
    _close(_gpu(*args, launches=2, form="SINGLE"), _reference(*args), "gpu T=%d H=%d L=%d B=%d" % (T, H, L, B))


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,L,B", [(1, 64, 1, 16), (3, 32, 1, 2), (4, 32, 4, 5), (5, 64, 2, 4), (4, 128, 4, 3), (7, 256, 3, 8),
                                     (3, 256, 2, 16), (3, 256, 4, 13), (5, 512, 2, 9), (4, 512, 3, 16), (3, 512, 4, 7), (3, 512, 1, 16),
                                     (5, 64, 1, 9), (6, 64, 2, 12), (5, 64, 4, 16), (7, 128, 1, 10), (5, 128, 2, 16), (6, 128, 3, 11), (5, 128, 4, 9),
                                     (5, 512, 2, 8), (6, 512, 3, 2), (5, 512, 1, 4), (5, 512, 1, 6)])
def test_rows_of_a_batch_share_a_step(T, H, L, B):
    """The form for several sequences: groups of four rows, full and ragged, one and two tiles of rows
    a workgroup, every depth, two to eight waves, more finishing (layer, tile) pairs than waves; two
    launches on one workspace."""
    args = _inputs(T + H + L + B, T, H, L, B)
    want, ran = _reference(*args), []
    # one tile of rows a workgroup and two, where the form is built and resident
    for form in ("ROWS", "ROWS2"):
        if form == "ROWS2" and (H < 512 or L == 4) or form == "ROWS" and H == 512 and (L == 4 or B > 8):
            continue
        _close(_gpu(*args, launches=2, form=form), want, "gpu %s T=%d H=%d L=%d B=%d" % (form, T, H, L, B))
        ran.append(form)
    if not ran:   # four layers of 512 units
        _close(_gpu(*args, launches=2, form="SINGLE"), want, "gpu T=%d H=%d L=%d B=%d" % (T, H, L, B))


@pytest.mark.gpu
def test_launches_in_a_row_on_one_workspace_and_no_initial_state():
    x, wih, whh, bih, bhh, _, _ = _inputs(21, 10, 128, 2, 2)
    z = torch.zeros(2, 2, 128)
    for form in ("SINGLE", "ROWS", "DIE"):
        _close(_gpu(x, wih, whh, bih, bhh, None, None, launches=3, form=form), _reference(x, wih, whh, bih, bhh, z, z), "third launch, " + form)


@pytest.mark.gpu
def test_benchmark_configuration_against_nn_lstm():
    """T = 64, H = 512, two layers, zero initial states: the library routine as a second opinion."""
    x, wih, whh, bih, bhh = oc.c4_inputs(0)
    z = torch.zeros(2, 1, 512)
    results = [_gpu(x, wih, whh, bih, bhh, z, z, form=form) for form in ("DIE", "SINGLE")]
    lstm = torch.nn.LSTM(512, 512, 2)
    with torch.no_grad():
        for l in range(2):
            getattr(lstm, "weight_ih_l%d" % l).copy_(wih[l].transpose(1, 2).reshape(2048, 512))
            getattr(lstm, "weight_hh_l%d" % l).copy_(whh[l].transpose(1, 2).reshape(2048, 512))
            getattr(lstm, "bias_ih_l%d" % l).copy_(bih[l].reshape(2048))
            getattr(lstm, "bias_hh_l%d" % l).copy_(bhh[l].reshape(2048))
        ref, (hn, cn) = lstm(x)
    for got in results:
        _close(got, (ref, hn, cn), "nn.LSTM")


@pytest.mark.gpu
def test_unsupported_shapes_are_refused():
    from functs_amd._lib import C, lib
    dev = torch.device("cuda:0")
    t = torch.zeros(1 << 16, device=dev)
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device=dev)
    p = t.data_ptr()
    rc = lib.fx_lstm_stack(p, p, p, p, p, p, p, p, p, p, 4, 1, 48, 2, ws.data_ptr(), 1 << 20, None)   # hidden not a multiple of 32
    assert rc == C["FX_E_UNSUPPORTED"]
    rc = lib.fx_lstm_stack(p, p, p, p, p, p, p, p, p, p, 4, 1, 64, 5, ws.data_ptr(), 1 << 20, None)   # five layers
    assert rc == C["FX_E_UNSUPPORTED"]


@pytest.mark.gpu
def test_a_form_that_is_not_built_for_the_sizes_is_refused():
    from functs_amd._lib import C, lib
    st = _Stack(4, 32, 2, 2)
    with lstm_form("DIE"):
        assert st.rc() == C["FX_E_UNSUPPORTED"]
    with lstm_form("ROWS2"):
        assert st.rc() == C["FX_E_UNSUPPORTED"]
    assert lib.fx_set_lstm_form(99) == C["FX_E_INVALID"] and lib.fx_set_lstm_form(-1) == C["FX_E_INVALID"]
    assert lib.fx_set_lstm_form(0) == 0
    st.launch()
    torch.cuda.synchronize()
    st.check("any form")
    assert lib.fx_lstm_form() == C["FX_LSTM_FORM_ROWS"]


def test_sizes_the_kernel_is_built_for():
    from functs_amd._lib import lib
    assert lib.fx_lstm_stack_fits(1, 512, 2) == 1 and lib.fx_lstm_stack_fits(16, 512, 4) == 1
    assert lib.fx_lstm_stack_fits(1, 1024, 2) == 1 and lib.fx_lstm_stack_fits(1, 1024, 3) == 0
    assert lib.fx_lstm_stack_fits(1, 96, 2) == 0 and lib.fx_lstm_stack_fits(17, 64, 2) == 0 and lib.fx_lstm_stack_fits(1, 64, 5) == 0


class _Stack:
    """One stack's operands and workspace on the device."""

    def __init__(self, T, H, L, B):
        from functs_amd._lib import lib
        self.dev, self.T, self.H, self.L, self.B = torch.device("cuda:0"), T, H, L, B
        args = _inputs(T + H + L + B, T, H, L, B)
        self.want = _reference(*args)
        self.args = [t.contiguous().to(self.dev) for t in args]
        self.ws = torch.zeros(lib.fx_lstm_stack_workspace_bytes(B, H, L), dtype=torch.uint8, device=self.dev)
        self.out = [torch.empty(T, B, H, device=self.dev)] + [torch.empty(L, B, H, device=self.dev) for _ in range(2)]

    def rc(self):
        from functs_amd._lib import lib
        return lib.fx_lstm_stack(*[t.data_ptr() for t in self.args + self.out], self.T, self.B, self.H, self.L, self.ws.data_ptr(),
                                 self.ws.numel(), ctypes.c_void_p(torch.cuda.current_stream(self.dev).cuda_stream))

    def launch(self):
        from functs_amd._lib import check
        check(self.rc())

    def check(self, what):
        _close(tuple(t.cpu() for t in self.out), self.want, what)


@pytest.fixture
def short_waits():
    """Waits that are given up after a fraction of a second."""
    from functs_amd._lib import lib
    lib.fx_set_lstm_spin_limit(100000)
    yield lib
    lib.fx_set_lstm_spin_limit(1000000)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[(12, 512, 2, 8), (9, 512, 2, 8)], [(12, 512, 2, 8), (12, 512, 2, 1), (12, 256, 1, 16)], [(12, 512, 2, 1)] * 4])
def test_launches_on_several_streams_take_turns_where_they_do_not_fit_together(sizes, short_waits):
    """Stacks that take the whole device, or together more than it, on a stream each: none starves."""
    stacks = [_Stack(*s) for s in sizes]
    streams = [torch.cuda.Stream() for _ in stacks]
    torch.cuda.synchronize()
    print("fx_lstm_stack on %d streams: %s" % (len(sizes), sizes), flush=True)
    for _ in range(4):
        for st, s in zip(stacks, streams):
            with torch.cuda.stream(s):
                st.launch()
                st.launch()
    torch.cuda.synchronize()
    assert short_waits.fx_async_error(1) == 0
    for st, s in zip(stacks, sizes):
        st.check("streams %r" % (s,))


@pytest.mark.gpu
@pytest.mark.parametrize("order", [(0, 1), (1, 0), (0, 1, 2, 0, 2, 1)])
def test_the_default_stream_takes_turns_with_others(order, short_waits):
    """The default stream's event is recorded when a launch on another one has to wait for it."""
    stacks = [_Stack(12, 512, 2, 8), _Stack(9, 512, 2, 8), _Stack(5, 512, 1, 16)]
    streams = [torch.cuda.default_stream(), torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    print("fx_lstm_stack on the default stream and others: %r" % (order,), flush=True)
    for _ in range(5):
        for i in order:
            with torch.cuda.stream(streams[i]):
                stacks[i].launch()
                stacks[i].launch()
    torch.cuda.synchronize()
    assert short_waits.fx_async_error(1) == 0
    for i in set(order):
        stacks[i].check("stream %d" % i)


@pytest.mark.gpu
def test_a_captured_launch_leaves_room_for_another(short_waits):
    """A graph's launch is replayed whenever the program likes: it and every later launch keep to half of
    the device, so a replay and a call on another stream run side by side; one workspace serves both forms."""
    a, b = _Stack(12, 512, 2, 8), _Stack(9, 512, 2, 8)
    side = torch.cuda.Stream()
    print("fx_lstm_stack captured", flush=True)
    a.launch()   # (the whole device, words)
    torch.cuda.synchronize()
    a.check("before the capture")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        a.launch()
    for _ in range(4):
        for t in a.out + b.out:
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        with torch.cuda.stream(side):
            b.launch()
        torch.cuda.synchronize()
        assert short_waits.fx_async_error(1) == 0
        a.check("replay")
        b.check("beside a replay")
    a.launch()
    torch.cuda.synchronize()
    a.check("a call on the graph's workspace")
    assert short_waits.fx_async_error(1) == 0
