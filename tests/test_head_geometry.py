"""Chunks and sub-tiles of the detection-head kernel (fx_head_geometry): the limits that the kernel is built for over
all sizes, few chunks to look back over, and no more of LDS than a chunk's rows take."""
import ctypes
import os
import subprocess

import pytest


@pytest.fixture(scope="module")
def geometry(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("head") / "libhead_geometry.so")
    src = os.path.join(os.path.dirname(os.path.abspath(__file__)), "support", "head_geometry.cpp")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", src, "-o", so])
    lib = ctypes.CDLL(so)

    def of(rows, tasks, S):
        out = (ctypes.c_uint32 * 4)()
        lib.fx_head_geometry_of(ctypes.c_uint32(rows), ctypes.c_uint32(tasks), ctypes.c_uint32(S), out)
        return tuple(out)
    return of


@pytest.mark.parametrize("S", [6, 7, 9, 10, 13, 18, 23, 24, 25, 31, 32, 45, 47, 48, 55, 64, 85, 96, 97, 300, 700])
def test_limits_of_the_kernel(geometry, S):
    for rows in (1, 5, 63, 64, 65, 127, 191, 192, 193, 255, 256, 257, 3087, 10647, 14175, 22743, 200000):
        for tasks in (1, 2, 4, 7, 9, 12, 16, 20, 64, 300):
            chunk, sub, carried, window = geometry(rows, tasks, S)
            assert 1 <= sub <= carried <= 256 and (carried * S + 6) <= 6 * 256 * 4, (rows, tasks)
            assert min(rows, 64) <= chunk <= 256, (rows, tasks)   # (the status words are allocated for chunks of 64 rows)
            assert sub <= max(chunk, 64) and window <= (max(chunk, 64) * S + 10) * 4, (rows, tasks)   # LDS for a chunk's rows only
            assert -(-chunk // sub) == -(-chunk // carried), (rows, tasks)   # as few rounds as the loads allow


def test_narrow_rows_are_looked_back_over_in_few_chunks(geometry):
    for rows, tasks, S in ((14175, 9, 10), (18207, 7, 10), (10647, 16, 12), (22743, 12, 13), (22743, 1, 13), (10647, 1, 18), (10647, 1, 85), (14175, 9, 65)):
        chunk, _, _, _ = geometry(rows, tasks, S)
        assert chunk >= 128 and -(-rows // chunk) <= 119


def test_a_small_launch_is_not_made_smaller(geometry):
    """An image of few rows keeps a workgroup for 64 of them: looking back over 64 chunks is one look."""
    assert geometry(3087, 1, 95)[0] == 64 and geometry(3087, 1, 10)[0] == 64
    assert geometry(6300, 4, 25)[0] == 99 and geometry(3087, 20, 25)[0] == 192


# chunks of 256, 192, 128 and 64 rows with last ones of a few, a chunk in one round of loads and in several
@pytest.mark.gpu
@pytest.mark.parametrize("rows,C,batch", [(14175, 5, 9), (14177, 4, 9), (10647, 13, 3), (193, 20, 2), (257, 7, 400), (130, 40, 1), (3087, 40, 2), (3089, 75, 5), (255, 91, 30)])
def test_every_geometry_against_the_two_passes(rows, C, batch):
    from functs_amd._lib import lib
    from tests.test_head_stream import _head, _inputs
    from tests.util import assert_exact, run_region
    batch = None if batch == 1 else batch
    args = _inputs(rows, C, batch or 1, seed=rows + C)
    one = run_region("hip", _head(batch=batch), *args)
    lib.fx_set_head_kernel(0)
    try:
        two = run_region("hip", _head(batch=batch), *args)
    finally:
        lib.fx_set_head_kernel(1)
    assert_exact(one, two, "rows=%d classes=%d batch=%s" % (rows, C, batch))
