"""GEMM tiles with a side of 192 (16 bits, fp8) where they can go wrong: one whole tile, tiles moved back in either direction, an odd
number of k-tiles, a moved-back k-tile, fewer k-tiles than LDS buffers, both weight layouts, both result types (16-bit results leave through
LDS as whole rows).  Small whole numbers: every sum is exact in fp32, and 16-bit results are its rounding."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(m, n, k, trans_b, batch=1):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m + 3 * n + 7 * k)
    lead = (batch,) if batch > 1 else ()
    a = torch.randint(-3, 4, lead + (m, k), generator=gen, device="cuda").float()
    b = torch.randint(-3, 4, lead + ((n, k) if trans_b else (k, n)), generator=gen, device="cuda").float()
    return a, b, a.double() @ (b.double().transpose(-1, -2).contiguous() if trans_b else b.double())


TILES = [(256, 192, 4, 2, 2), (192, 256, 2, 4, 2), (128, 192, 4, 2, 2), (128, 192, 4, 2, 3), (192, 128, 2, 4, 2), (192, 128, 2, 4, 3)]


def _sizes(bm, bn):
    return [(bm, bn, 64), (bm + 1, bn + 8, 192), (2 * bm - 3, 3 * bn - 16, 200), (bm + 100, 2 * bn, 1096), (700, 1000, 640)]


def _tile(bm, bn, wm, wn, nbuf):
    return dict(BM=bm, BN=bn, WM=wm, WN=wn, NBUF=nbuf, M16=1, D2L=1)


@pytest.fixture(scope="module")
def compiled():
    """The kernels of test_16_bit: one after the other they are most of its time."""
    from compile_ahead import compile_ahead
    compile_ahead([("gemm_bf16", dict(M=m, N=n, K=k, BATCH=1, TA=0, TB=tb, OUT_BF16=out, ALIGN=16, **(dict(F16=1) if half else {}), **_tile(*tile)))
                   for tile in TILES for m, n, k in _sizes(*tile[:2]) for tb in (0, 1) for half in (0, 1) for out in (0, 1)])


@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("bm,bn,wm,wn,nbuf", TILES)
def test_16_bit(bm, bn, wm, wn, nbuf, trans_b, compiled):
    from kernelcodegen_amd import ops
    cfg = _tile(bm, bn, wm, wn, nbuf)
    for m, n, k in _sizes(bm, bn):
        a, b, ref = _operands(m, n, k, trans_b)
        for dtype in (torch.bfloat16, torch.float16):
            for out in (torch.float32, dtype):
                c = ops.batched_matmul(a.to(dtype), b.to(dtype), trans_b=trans_b, out_dtype=out, **cfg)
                assert torch.equal(c, ref.float().to(out)), (m, n, k, dtype, out)
    a, b, ref = _operands(bm + 5, bn + 16, 256, trans_b, 3)
    assert torch.equal(ops.batched_matmul(a.bfloat16(), b.bfloat16(), trans_b=trans_b, **cfg), ref.float())


@pytest.mark.parametrize("trans_b", [True, False])
def test_fp8(trans_b):
    from kernelcodegen_amd import ops
    for m, n, k in [(256, 192, 128), (257, 208, 256), (511, 560, 384), (600, 384, 1152), (1000, 1008, 640)]:
        a, b, ref = _operands(m, n, k, trans_b)
        for out in (torch.float32, torch.bfloat16):
            c = ops.matmul_fp8(a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn), 0.5, 4.0, trans_b=trans_b, out_dtype=out, BM=256, BN=192, WM=4, WN=2)
            assert torch.equal(c, (2 * ref).float().to(out)), (m, n, k, out)


@pytest.mark.parametrize("m,n,k,dtype", [(1000, 11008, 512, "bf16"), (400, 11008, 1024, "f16"), (1500, 2816, 1024, "bf16"), (1500, 11008, 512, "fp8"), (700, 11008, 2048, "fp8")])
@pytest.mark.parametrize("trans_b", [True, False])
def test_chosen(m, n, k, dtype, trans_b):
    """The same without asking for a tile: the rule picks one for these sizes."""
    from kernelcodegen_amd import ops, runtime as R
    family = "gemm_fp8" if dtype == "fp8" else "gemm_bf16"
    text = R.emit_kernel(family, **R.launch_params(family, dict(M=m, N=n, K=k, TB=int(trans_b), ALIGN=16, F16=int(dtype == "f16"), OUT_BF16=1)))[0]
    assert any("#define %s 192\n" % name in text for name in ("GB_BM", "GB_BN", "G8_BN"))
    a, b, ref = _operands(m, n, k, trans_b)
    if dtype == "fp8":
        c = ops.matmul_fp8(a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn), 1.0, 1.0, trans_b=trans_b, out_dtype=torch.bfloat16)
    else:
        t = torch.bfloat16 if dtype == "bf16" else torch.float16
        c = ops.batched_matmul(a.to(t), b.to(t), trans_b=trans_b, out_dtype=t)
    assert torch.equal(c, ref.float().to(c.dtype))


@pytest.mark.parametrize("m,n,k,batch", [(70000, 176, 640, 1), (65793, 16, 128, 1), (65793, 48, 384, 1), (256, 128, 512, 256), (300, 144, 384, 150)])
def test_fp8_of_fewer_columns(m, n, k, batch):
    """Row-major weights of fewer than 192 columns: the same tiles on the guarded kernel."""
    from kernelcodegen_amd import ops, runtime as R
    text = R.emit_kernel("gemm_fp8", **R.launch_params("gemm_fp8", dict(M=m, N=n, K=k, TB=0, BATCH=batch, ALIGN=16, OUT_BF16=1)))[0]
    assert "#define GF_BN 192\n" in text and "#define GF_EDGE 1\n" in text
    a, b, ref = _operands(m, n, k, False, batch)
    for out in (torch.float32, torch.bfloat16):
        c = ops.matmul_fp8(a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn), 0.5, 4.0, trans_b=False, out_dtype=out)
        assert torch.equal(c, (2 * ref).float().to(out)), out
