"""Softmax rows that start anywhere: lengths that no vector divides, from fewer lanes than values in front of the first vector boundary to
rows that fill the registers, operands on every element offset, in place, and the rows next to each row untouched."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPE = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
# relative.  fp32: the exponent (x - max) log2(e) is up to 40 in size (values within 27 of each other) and rounded twice, 2^-24 of it
# each time, which the exponential turns into 40 * 2 * 2^-24 * ln 2 = 3.3e-6; the hardware's exp2, the sum and the quotient add a few
# 2^-24.  16 bits: half a unit in the last place of the result on top, 2^-8 of it (bf16, 8 significant bits) or 2^-11 (half, 11).
TOL = {"f32": 5e-6, "bf16": 2.0 ** -8 + 1e-5, "f16": 2.0 ** -11 + 1e-5}


@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("rows,n", [(4200, 257), (4100, 1023), (1100, 1025), (1030, 2047), (530, 2049), (300, 4095), (260, 8191), (70, 16383), (33, 32001), (1100, 1021), (2100, 514)])
def test_rows_start_anywhere(rows, n, dtype, inplace):
    from kernelcodegen_amd import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    for off in (0, 1, 3, 5):
        buf = (torch.randn(rows * n + 32, generator=gen, device="cuda") * 3).to(DTYPE[dtype])
        x = buf[8 + off:8 + off + rows * n].view(rows, n)
        want = torch.softmax(x.double(), -1)
        before = buf.clone()
        y = ops.softmax(x, inplace=inplace)
        # (16-bit results below the smallest normal number round to its multiples)
        small = {"f16": 2.0 ** -25, "bf16": 0.0, "f32": 0.0}[dtype]
        assert bool(((y.double() - want).abs() <= TOL[dtype] * want + small + 1e-37).all()), (rows, n, off)
        if inplace:
            assert y.data_ptr() == x.data_ptr()
            assert torch.equal(buf[:8 + off], before[:8 + off]) and torch.equal(buf[8 + off + rows * n:], before[8 + off + rows * n:])
        else:
            assert torch.equal(buf, before)
