"""A sequence's layers on one die (fx_lstm_die_kernel): the schedule, the ring between stages and the tags on
host threads, and the kernel against the oracle.  Tolerances as for the other forms of fx_lstm_stack
(tests/test_lstm_kernel.py)."""
import ctypes
import os
import subprocess

import pytest
import torch

from tests.test_lstm_kernel import _close, _gpu, _inputs, _reference, lstm_form


@pytest.fixture(scope="module")
def emul(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("lstm_die") / "liblstm_die_emul.so")
    src = os.path.join(os.path.dirname(os.path.abspath(__file__)), "support", "lstm_die_emul.cpp")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-pthread", src, "-o", so])
    lib = ctypes.CDLL(so)
    lib.fx_lstm_die_emul.argtypes = [ctypes.c_void_p] * 10 + [ctypes.c_int] * 5 + [ctypes.c_uint32, ctypes.c_int, ctypes.c_uint32, ctypes.c_int, ctypes.c_int]
    lib.fx_lstm_die_emul_give_up.argtypes = [ctypes.c_void_p] * 10 + [ctypes.c_int] * 5 + [ctypes.c_uint32] + [ctypes.c_int] * 3
    lib.fx_lstm_others_emul.argtypes = [ctypes.c_int] * 2 + [ctypes.c_uint32] * 2 + [ctypes.c_int]
    return lib


def _run(lib, args, n_wg=4, launches=1, base0=0, slow=(-1, -1), spin=1 << 30):
    T, B, H = args[0].shape
    L = args[1].size(0)
    out, sh, sc = torch.zeros(T, B, H), torch.zeros(L, B, H), torch.zeros(L, B, H)
    ts = [t.contiguous() for t in args]
    rc = lib.fx_lstm_die_emul(*[t.data_ptr() for t in ts + [out, sh, sc]], T, B, H, L, n_wg, spin, launches, base0, *slow)
    return (out, sh, sc), rc


# one and two stages of two layers, stages of one layer whose rings go round more than twice
@pytest.mark.parametrize("T,H,L,B,launches", [(1, 64, 1, 1, 3), (1, 64, 4, 2, 2), (2, 128, 3, 2, 2), (7, 64, 2, 3, 3), (20, 256, 4, 1, 2), (40, 512, 2, 1, 1), (1, 512, 3, 1, 3)])
def test_schedule_and_ring_on_host_threads(emul, T, H, L, B, launches):
    args = _inputs(T + H + L, T, H, L, B)
    got, rc = _run(emul, args, launches=launches)
    assert rc == 0
    _close(got, _reference(*args), "emul T=%d H=%d L=%d B=%d" % (T, H, L, B))


@pytest.mark.parametrize("slow", [(0, 1), (1, 0), (2, 3)])
def test_a_stage_that_lags_is_not_overrun(emul, slow):
    """One workgroup of the first, second or third stage dawdles: the ring holds the stage before it up."""
    args = _inputs(3, 45, 512, 3, 1)
    got, rc = _run(emul, args, slow=slow)
    assert rc == 0
    _close(got, _reference(*args), "slow %r" % (slow,))


def test_tags_start_over_before_they_wrap(emul):
    args = _inputs(4, 5, 512, 2, 1)
    got, rc = _run(emul, args, launches=3, base0=0x80000000 - 8)
    assert rc == 0
    _close(got, _reference(*args), "after the tags were cleared")


# a stage's own h, the ring to the next stage (whose reader or writer is gone), and the three areas of a workspace
@pytest.mark.parametrize("H,L,B,stop,marked", [(64, 2, 1, (0, 1), 0), (64, 2, 2, (0, 0), 1), (512, 3, 1, (0, 2), 2), (512, 3, 1, (1, 0), 0), (512, 2, 2, (1, 3), 1), (256, 4, 1, (1, 1), 2)])
def test_a_wait_that_cannot_end_is_given_up_and_its_workspace_refused(emul, H, L, B, stop, marked):
    args = [t.contiguous() for t in _inputs(H + L, 40, H, L, B)]
    out, sh, sc = torch.zeros(40, B, H), torch.zeros(L, B, H), torch.zeros(L, B, H)
    bits = emul.fx_lstm_die_emul_give_up(*[t.data_ptr() for t in args + [out, sh, sc]], 40, B, H, L, 4, 3000, *stop, marked)
    for bit, what in ((1, "the launch with a workgroup less did not give up"), (2, "it left values that look like results"),
                      (4, "the workspace of a given-up wait was used again"), (8, "and its results are no NaN"),
                      (16, "a launch that another form's error word refuses ran"), (32, "and its results are no NaN"), (64, "the cleared workspace failed")):
        assert bits & bit, what
    _close((out, sh, sc), _reference(*args), "on the cleared workspace")


def test_streams_that_launched_lately_are_told_apart(emul):
    others = emul.fx_lstm_others_emul
    for device in (1 << 20, 64):      # launches that overlap, launches that take turns
        assert others(1, 5, 64, device, 0) == 0
        assert others(2, 0, 64, device, 0) == others(2, 62, 64, device, 0) == 1
        assert others(2, 64, 64, device, 0) == 0    # stream 1 launched 64 launches ago
        assert others(1, 5, 64, device, 7) == 1     # a second stream's first launch


# sizes whose workgroups, spread over the chip, take at most half of it; (5, 64, 3, 8): fewer steps than the kernel is taken for
@pytest.mark.gpu
@pytest.mark.parametrize("T,H,L,B", [(9, 64, 2, 1), (12, 64, 3, 8), (5, 64, 3, 8), (6, 128, 3, 8), (6, 128, 4, 3), (7, 256, 3, 4), (9, 256, 4, 2), (20, 512, 2, 1), (8, 512, 4, 1), (6, 512, 1, 4)])
def test_a_captured_stack_computes_what_the_calls_beside_it_compute(T, H, L, B):
    """To the bit, whether or not another stream has launched stacks lately."""
    from functs_amd import jit as fj
    from functs_amd._lib import C, lib
    from functs_amd.benchmark import PROGRAMS
    from oracle import configs as oc
    args = oc.c4_inputs(3, T, H, L, B)
    gpu = [a.cuda() if isinstance(a, torch.Tensor) else a for a in args]
    form = C["FX_LSTM_FORM_ROWS" if (T, H) == (5, 64) else "FX_LSTM_FORM_SPREAD"]
    eager = fj.build(fj.script(PROGRAMS["c4"]), list(args))
    for other in (False, True):
        if other:
            with torch.cuda.stream(torch.cuda.Stream()):
                eager(*gpu)
            torch.cuda.synchronize()
        graphed = fj.build(fj.script(PROGRAMS["c4"]), list(args), hip_graph=True)
        graphed(*gpu)
        assert lib.fx_lstm_form() == form
        for _ in range(3):
            want = eager(*gpu)
            torch.cuda.synchronize()
            for g, w in zip(graphed(*gpu), want):
                assert torch.equal(g, w), "after launches on another stream: %s" % other
    with torch.cuda.stream(torch.cuda.Stream()):   # and beside the other stream's
        beside = eager(*gpu)
        assert lib.fx_lstm_form() == form
    torch.cuda.synchronize()
    assert all(torch.equal(b, w) for b, w in zip(beside, want))


@pytest.mark.gpu
def test_a_pinned_form_gives_the_same_bits_to_calls_and_captures():
    """Sizes whose workgroups on dies take the whole device: calls and captures differ in form, unless one is asked for."""
    from tests.test_lstm_kernel import _Stack
    from functs_amd._lib import C, lib
    st = _Stack(9, 256, 3, 8)
    with lstm_form("ROWS"):
        st.launch()
        torch.cuda.synchronize()
        call = [t.clone() for t in st.out]
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            st.launch()
    for t in st.out:
        t.fill_(float("nan"))
    g.replay()
    torch.cuda.synchronize()
    assert lib.fx_async_error(1) == 0
    st.check("replay")
    assert all(torch.equal(a, b) for a, b in zip(call, st.out))
    for form in ("DIE", "SPREAD"):   # (in a capture these would starve a second replay)
        with lstm_form(form):
            st.launch()
            torch.cuda.synchronize()
            st.check(form)
            with torch.cuda.graph(torch.cuda.CUDAGraph()):
                torch.zeros(1, device="cuda")
                assert st.rc() == C["FX_E_UNSUPPORTED"]


@pytest.mark.gpu
def test_small_stacks_on_many_streams_and_replays_hold_little():
    """Three graphs of small stacks at once beside calls on three streams: a launch that is not alone claims the
    workgroups that it has, on no die in particular."""
    from tests.test_lstm_kernel import _Stack
    from functs_amd._lib import C, lib
    stacks = [_Stack(12, 64, 1, 1) for _ in range(6)]
    graphs, streams = [], [torch.cuda.Stream() for _ in stacks]
    torch.cuda.synchronize()
    print("fx_lstm_stack on six streams", flush=True)
    for st in stacks[:3]:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            st.launch()
        assert lib.fx_lstm_form() == C["FX_LSTM_FORM_SPREAD"]
        graphs.append(g)
    for _ in range(5):
        for i, (st, s) in enumerate(zip(stacks, streams)):
            with torch.cuda.stream(s):
                graphs[i].replay() if i < 3 else st.launch()
    torch.cuda.synchronize()
    assert lib.fx_async_error(1) == 0
    for st in stacks:
        st.check("side by side")


# every width and depth of a stage, one to eight sequences, rings that go round, shorter sequences than the lag
@pytest.mark.gpu
@pytest.mark.parametrize("T,H,L,B", [(1, 64, 1, 1), (2, 64, 3, 8), (33, 64, 4, 5), (1, 128, 4, 8), (19, 128, 2, 3), (1, 256, 1, 8), (30, 256, 3, 8),
                                     (50, 256, 4, 4), (21, 256, 2, 1), (1, 512, 3, 2), (3, 512, 2, 4), (70, 512, 2, 4), (40, 512, 4, 2), (9, 512, 1, 8)])
def test_kernel_against_the_oracle(T, H, L, B):
    args = _inputs(T + H + L + B, T, H, L, B)
    want, got = _reference(*args), _gpu(*args, launches=3, form="DIE")
    _close(got, want, "gpu T=%d H=%d L=%d B=%d" % (T, H, L, B))
    # spread over the dies, where values go by the memory side: the same sums in the same order
    spread = _gpu(*args, launches=3, form="SPREAD")
    _close(spread, want, "gpu, spread, T=%d H=%d L=%d B=%d" % (T, H, L, B))
    assert all(torch.equal(a, b) for a, b in zip(got, spread))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["DIE", "SPREAD"])
@pytest.mark.parametrize("H,L,B", [(64, 1, 1), (256, 3, 2), (256, 4, 2), (512, 2, 1)])
def test_a_given_up_wait_ends_the_kernel_and_marks_the_workspace(H, L, B, form):
    from tests.test_lstm_kernel import _Stack
    from functs_amd._lib import C, lib
    st = _Stack(20, H, L, B)
    with lstm_form(form):
        # a wait is given up at its first look without a value; a launch whose every look finds one is right, and another is made
        lib.fx_set_lstm_spin_limit(0)
        try:
            for _ in range(20):
                st.launch()
                torch.cuda.synchronize()
                error = lib.fx_async_error(1)
                if error != 0:
                    break
                st.check("no wait was given up")
        finally:
            lib.fx_set_lstm_spin_limit(1000000)
        assert error == C["FX_ASYNC_BARRIER"] and bool(st.out[0][-1].isnan().all())
        st.launch()   # refused
        torch.cuda.synchronize()
        assert lib.fx_async_error(1) == C["FX_ASYNC_BARRIER"] and all(bool(t.isnan().all()) for t in st.out)
        st.ws.zero_()
        st.launch()
        torch.cuda.synchronize()
        assert lib.fx_async_error(1) == 0
        st.check("on the cleared workspace")


@pytest.mark.gpu
def test_operands_of_any_float_alignment():
    from functs_amd._lib import check, lib
    args = _inputs(8, 6, 256, 2, 2)
    odd = [torch.cat([t.new_zeros(1), t.reshape(-1)]).cuda()[1:] for t in args]
    assert all(t.data_ptr() % 16 == 4 for t in odd)
    T, B, H, L = 6, 2, 256, 2
    n = lib.fx_lstm_stack_workspace_bytes(B, H, L)
    ws = torch.zeros(n, dtype=torch.uint8, device="cuda")
    out = [torch.empty(T, B, H, device="cuda"), torch.empty(L, B, H, device="cuda"), torch.empty(L, B, H, device="cuda")]
    with lstm_form("DIE"):
        check(lib.fx_lstm_stack(*[t.data_ptr() for t in odd + out], T, B, H, L, ws.data_ptr(), n, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    assert lib.fx_async_error(1) == 0
    _close([t.cpu() for t in out], _reference(*args), "odd alignment")


# either side of the fewest steps that the kernel is taken for, whatever else the process has launched or captured
@pytest.mark.gpu
@pytest.mark.parametrize("T,H,L,B,other", [(1, 64, 1, 1, "SINGLE"), (2, 64, 1, 1, None), (3, 64, 2, 4, "ROWS"), (4, 64, 2, 4, None), (6, 64, 3, 8, "ROWS"),
                                           (7, 64, 3, 8, None), (2, 128, 2, 3, "ROWS"), (3, 128, 2, 3, None), (4, 128, 3, 8, "ROWS"), (5, 128, 3, 8, None),
                                           (4, 256, 3, 4, "ROWS"), (5, 256, 3, 4, None), (1, 256, 4, 2, None), (5, 512, 1, 4, "SPREAD"), (23, 512, 1, 1, "SPREAD"),
                                           (9, 512, 2, 1, "SPREAD"), (19, 512, 2, 2, "SPREAD"), (1, 512, 3, 1, "SPREAD")])
def test_short_sequences_take_the_forms_that_start_sooner(T, H, L, B, other):
    from functs_amd._lib import C, lib
    args = _inputs(T + H + L + B, T, H, L, B)
    _close(_gpu(*args, launches=2), _reference(*args), "T=%d H=%d L=%d B=%d" % (T, H, L, B))
    assert lib.fx_lstm_form() in ([C["FX_LSTM_FORM_" + other]] if other else [C["FX_LSTM_FORM_DIE"], C["FX_LSTM_FORM_SPREAD"]])
