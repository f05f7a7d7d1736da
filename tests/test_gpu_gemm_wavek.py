"""Products whose wavefronts split k (kernels/gemm_wavek.hip), at the sizes where they can go wrong: rows, columns and steps of k
that the tile, the 128-byte step and the wavefronts do not divide, one row, fewer rows than a group of eight, batches.

Operands are small whole numbers, so every order of summation gives the same fp32 sum (below 2^24) and results are compared exactly;
one column has an infinity as its last value of k, which must reach that column alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPE = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "fp8": torch.float8_e4m3fn}


def _check(dtype, m, n, k, trans_b, batch, out, cfg):
    from kernelcodegen_amd import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m * 31 + n * 7 + k)
    lead = (batch,) if batch > 1 else ()
    a = torch.randint(-3, 4, lead + (m, k), generator=gen, device="cuda").float()
    b = torch.randint(-3, 4, lead + ((n, k) if trans_b else (k, n)), generator=gen, device="cuda").float()
    ref = a.double() @ (b.double().transpose(-1, -2).contiguous() if trans_b else b.double())
    col = n // 2
    if dtype != "fp8":                    # e4m3 has no infinity
        if trans_b:
            b[..., col, k - 1] = float("inf")
        else:
            b[..., k - 1, col] = float("inf")
        last = a[..., k - 1]
        ref[..., col] = torch.where(last == 0, float("nan"), last.double() * float("inf"))
    if dtype == "fp8":
        c = ops.matmul_fp8(a.to(DTYPE[dtype]), b.to(DTYPE[dtype]), 0.5, 2.0, trans_b=trans_b, out_dtype=out, **cfg)
    else:
        c = ops.batched_matmul(a.to(DTYPE[dtype]), b.to(DTYPE[dtype]), trans_b=trans_b, out_dtype=out, **cfg)
    want = ref.to(torch.float32).to(out)
    assert torch.equal(torch.nan_to_num(c.float(), nan=1e30), torch.nan_to_num(want.float(), nan=1e30))


# tiles (rows, columns), wavefronts, steps in flight
FORMS = [(1, 1, 4, 1), (1, 2, 8, 2), (2, 4, 4, 2), (4, 4, 8, 1)]


@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16", "fp8"])
@pytest.mark.parametrize("form", FORMS)
def test_forms(form, dtype, trans_b):
    tm, tn, wk, depth = form
    es = DTYPE[dtype].itemsize
    if dtype == "fp8" and not trans_b and tn == 1:
        pytest.skip("a row-major fp8 load takes two columns and more")
    sizes = [(1, 64, 512 * 4 // es, 1), (7, 80, 528 * 4 // es, 3), (33, 80, 1040 * 2 // es, 1), (65, 48, 128 // es * wk + 16 // es, 2)]
    if dtype == "f32":
        sizes += [(40, 77, 333, 2), (9, 33, 1025, 1), (16, 16, 32 * wk + 3, 1)]
    outs = {"f32": [torch.float32], "f16": [torch.float16], "bf16": [torch.bfloat16, torch.float32], "fp8": [torch.bfloat16, torch.float32]}[dtype]
    for m, n, k, batch in sizes:
        cfg = dict(TM=tm, TN=tn, WAVEK=wk, DEPTH=depth)
        if not trans_b:
            cfg["VW"] = 1 if n % min(tn, 4) else min(tn, 4)
        for out in outs:
            _check(dtype, m, n, k, trans_b, batch, out, cfg)


@pytest.mark.parametrize("dtype,m,n,k,trans_b,batch", [
    ("bf16", 8, 1024, 4096, True, 1), ("f16", 1, 512, 512, False, 1), ("bf16", 33, 528, 1000, True, 1), ("f16", 48, 1600, 2056, False, 1),
    ("bf16", 200, 1024, 4096, True, 1), ("fp8", 16, 2048, 2048, True, 1), ("fp8", 3, 1040, 2064, False, 1), ("fp8", 64, 4096, 4096, False, 1),
    ("f32", 256, 256, 256, False, 1), ("f32", 257, 300, 771, True, 1), ("f32", 300, 301, 2001, False, 3), ("f32", 300, 304, 402, False, 2)])
def test_chosen(dtype, m, n, k, trans_b, batch):
    """The same without asking for a form: the rule picks it for these sizes."""
    from kernelcodegen_amd import runtime as R
    family = {"f32": "gemm_f32", "fp8": "gemm_fp8"}.get(dtype, "gemm_bf16")
    params = dict(M=m, N=n, K=k, BATCH=batch, TB=int(trans_b), ALIGN=16, OUT_BF16=int(dtype != "f32"), F16=int(dtype == "f16"))
    text, _ = R.emit_kernel(family, **R.launch_params(family, params))
    assert "#define GW_WK" in text
    out = {"f32": torch.float32, "f16": torch.float16}.get(dtype, torch.bfloat16)
    _check(dtype, m, n, k, trans_b, batch, out, {})
