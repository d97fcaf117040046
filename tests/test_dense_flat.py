"""Elementwise outputs whose operand lies as the output does are one long row (fx_lower.cpp).  Every layout gives what eager
mode gives, whether or not it is taken as one row."""
import pytest
import torch

from functs_amd.region import Region
from tests.util import run_region

# (shape of the memory, view of it as the operand): in order, of odd lengths, with extents of one, strided, transposed, broadcast, offset
LAYOUTS = {
    "2d": ((37, 53), lambda m: m),
    "rows_of_1": ((41, 1), lambda m: m),
    "one_row": ((1, 43), lambda m: m),
    "3d": ((3, 5, 7), lambda m: m),
    "ones_inside": ((6, 1, 9), lambda m: m),
    "4d": ((2, 3, 1, 5), lambda m: m),
    "part_of_rows": ((11, 24), lambda m: m[:, 3:16]),
    "every_second_row": ((22, 9), lambda m: m[::2]),
    "every_second_element": ((10, 26), lambda m: m[:, ::2]),
    "transposed": ((19, 33), lambda m: m.t()),
    "middle_transposed": ((3, 8, 5), lambda m: m.transpose(0, 1)),
    "broadcast_rows": ((1, 29), lambda m: m.expand(17, 29)),
    "broadcast_elements": ((17, 1), lambda m: m.expand(17, 31)),
    "offset": ((8, 40), lambda m: m[2:]),
}


def _region(rank, dtype):
    r = Region()
    x = r.tensor_input(dtype, rank)
    r.output(x * 2.0 + 1.0 if dtype is torch.float32 else x + 1)
    return r.finalize()


@pytest.mark.parametrize("backend", ["emul", pytest.param("hip", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("dtype", [torch.float32, torch.int32])
def test_layouts(backend, layout, dtype):
    shape, view = LAYOUTS[layout]
    n = 1
    for s in shape:
        n *= s
    x = view((torch.arange(n) % 8191).to(dtype).view(shape))
    print("flat", layout, dtype, flush=True)
    (got,) = run_region(backend, _region(x.dim(), dtype), x)
    assert torch.equal(got, x * 2.0 + 1.0 if dtype is torch.float32 else x + 1)


# outputs of some megabytes, of odd lengths and with operands that are not one row
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,rows,cols", [(torch.float32, 1023, 1025), (torch.float32, 1025, 1023), (torch.float32, 4099, 513),
                                             (torch.bfloat16, 2049, 1023), (torch.bfloat16, 2047, 1025), (torch.float16, 3001, 1111)])
def test_large_outputs_in_the_loop_program(dtype, rows, cols):
    import functs_amd.jit as fj
    from functs_amd.benchmark import PROGRAMS
    b = torch.randn(rows, cols + 3, device="cuda").to(dtype)
    for part in (b[:, :cols].contiguous(), b[:, :cols]):
        fn = fj.build(fj.script(PROGRAMS["c1"]), [part[:1].clone(), part, rows])
        print("large", dtype, rows, cols, part.is_contiguous(), flush=True)
        assert torch.equal(fn(part[:1].clone(), part, rows), part + 1)
