"""16-bit elements move as whole lane groups (one 64-bit access of 2-byte alignment per lane): values
against stock PyTorch, which rounds every operation, so one operation per region and exact results."""
import pytest
import torch

from functs_amd import Region
from tests.util import run_region

DTYPES = [torch.float16, torch.bfloat16]


def _same(got, ref):
    assert got.dtype == ref.dtype and got.shape == ref.shape
    n, m = torch.isnan(got), torch.isnan(ref)
    assert torch.equal(n, m) and torch.equal(got[~n].view(torch.int16), ref[~m].view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,cols,lo", [(1, 1, 0), (1, 3, 1), (5, 4, 0), (3, 257, 3), (64, 64, 1), (1025, 4096, 0), (1027, 4099, 5)])
def test_one_operation(dtype, rows, cols, lo):
    # (lo: the first column of a wider matrix, so that groups start at every 2-byte boundary)
    g = torch.Generator().manual_seed(cols)
    wide = (torch.randn(rows, cols + 8, generator=g) * 100).to(dtype)
    wide.view(-1)[:: 97] = float("nan")
    wide.view(-1)[1:: 89] = float("inf")
    wide.view(-1)[2:: 83] = torch.finfo(dtype).min
    x = wide[:, lo:lo + cols]
    r = Region()
    a = r.tensor_input(dtype, 2)
    r.output(a + 1.0)
    r.output(a.transpose(0, 1) * 3.0)      # (no consecutive loads)
    r.finalize()
    one, three = run_region("hip", r, x)
    _same(one, x + 1.0)
    _same(three, x.t() * 3.0)


# Whole groups are rounded two values at a time, the rest one by one (fx_bf16_pair, fx_bf16): every upper half of a float with lower
# halves below, at and above a tie.  Subnormal results, results that round up to infinity and every kind of NaN are among them.
@pytest.mark.gpu
@pytest.mark.parametrize("cols", [3, 4, 6, 4096])
def test_bfloat16_rounding_of_every_upper_half(cols):
    low = torch.tensor([0, 1, 0x7fff, 0x8000, 0x8001, 0xffff, 0x8000, 0x4000], dtype=torch.int64)
    bits = (torch.arange(1 << 16).view(-1, 1) << 16 | low).view(-1)
    bits = bits[:bits.numel() // (2 * cols) * 2 * cols].to(torch.uint32).view(torch.float32)
    x = torch.cat([bits, bits.flip(0)]).view(-1, cols)      # (either place of a pair)
    r = Region()
    a = r.tensor_input(torch.float32, 2)
    r.output(a.to(torch.bfloat16))
    r.finalize()
    (got,) = run_region("hip", r, x)
    _same(got, x.to(torch.bfloat16))
