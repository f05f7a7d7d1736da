"""Attention whose wavefronts split the keys (kernels/fmha_wavek.hip) at the sizes where it can go wrong: sequences that 32-key
tiles, query blocks and the wavefronts do not divide, one tile, wavefronts without a tile, both masks, every operand type.

The reference is fp64.  Tolerances, relative in the 2-norm: fp32 4e-6, a sum of up to 300 fp32 products with the hardware's exp2
(2e-7 each); 16 bits: half a unit in the last place of the probabilities and of the result, at most 2^-8 of a value (bf16)
or 2^-11 (half): both together 7.8e-3 and 9.8e-4."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPE = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
TOL = {"f32": 4e-6, "bf16": 8e-3, "f16": 1e-3}


def _reference(q, k, v, causal, scale):
    s = q.double() @ k.double().transpose(-1, -2).contiguous() * scale
    if causal:
        n = s.shape[-1]
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    return torch.softmax(s, -1) @ v.double()


def _check(b, h, s, d, dtype, causal, cfg, out=None, spread=1.0):
    from kernelcodegen_amd import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(s * 5 + d)
    q, k, v = (torch.randn(b, h, s, d, generator=gen, device="cuda").to(DTYPE[dtype]) for _ in range(3))
    # the largest score comes late and far above the others: the reference of the exponentials has to move
    k = (k.float() * torch.linspace(0.2, spread, s, device="cuda").view(1, 1, s, 1)).to(DTYPE[dtype])
    got = ops.fmha(q, k, v, causal=causal, out_dtype=out, **cfg)
    want = _reference(q, k, v, causal, d ** -0.5)
    assert got.dtype == (out or DTYPE[dtype])
    rel = float((got.double() - want).norm() / want.norm())
    assert rel < TOL[dtype], (s, d, cfg, rel)


FORMS = [dict(WAVEK=2), dict(WAVEK=4), dict(WAVEK=8), dict(WAVEK=4, QB=2), dict(WAVEK=1)]


TYPES = [("f32", 64), ("f32", 128), ("bf16", 64), ("f16", 64), ("bf16", 128), ("f16", 128), ("f16", 32), ("f32", 32)]
SIZES = [(1, 3, 1), (1, 8, 32), (2, 4, 33), (1, 5, 97), (1, 8, 300)]


@pytest.fixture(scope="module")
def compiled():
    """The kernels of test_forms: one after the other they are most of its time."""
    from compile_ahead import compile_ahead
    kernels = []
    for dtype, d in TYPES:
        for form in FORMS:
            for causal in (0, 1):
                for b, h, s in SIZES + [(1, 2, 130)]:
                    problem = dict(B=b, H=h, S=s, D=d, CAUSAL=causal, SCALE=d ** -0.5, FILL=1, **form)
                    if dtype == "f32":
                        if d < 128 or form["WAVEK"] <= 4:
                            kernels.append(("fmha_f32", problem))
                    else:
                        kernels += [("fmha_bf16", dict(problem, F16=int(dtype == "f16"), OUT_BF16=out)) for out in ((1, 0) if s == 130 else (1,))]
    compile_ahead(kernels)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype,d", TYPES)
@pytest.mark.parametrize("form", FORMS)
def test_forms(form, dtype, d, causal, compiled):
    if dtype == "f32" and d == 128 and form["WAVEK"] > 4:
        pytest.skip("the wavefronts' tiles do not fit the LDS")
    for b, h, s in SIZES:
        _check(b, h, s, d, dtype, causal, form)
    _check(1, 2, 130, d, dtype, causal, form, spread=40.0)
    if dtype != "f32":
        _check(1, 2, 130, d, dtype, causal, form, out=torch.float32)


@pytest.mark.parametrize("dtype,d,b,h,s,causal", [("bf16", 64, 1, 8, 333, False), ("f16", 128, 2, 16, 100, True), ("bf16", 128, 1, 8, 1024, True),
                                                  ("f32", 64, 2, 16, 512, False), ("f32", 128, 1, 12, 77, True), ("f16", 64, 1, 8, 2048, False)])
def test_chosen(dtype, d, b, h, s, causal):
    """The same without asking for a form: the rule picks it for these launches."""
    from kernelcodegen_amd import runtime as R
    family = "fmha_f32" if dtype == "f32" else "fmha_bf16"
    params = dict(B=b, H=h, S=s, D=d, CAUSAL=int(causal), SCALE=d ** -0.5, FILL=1)
    assert "#define FW_WK" in R.emit_kernel(family, **R.launch_params(family, params))[0]
    _check(b, h, s, d, dtype, causal, {})


def test_infinities_and_nan_stay_in_their_rows():
    """A key row of -inf scores takes no part; a NaN in one query's row reaches that row alone; +inf scores give NaN as the kernels of
    whole tiles do."""
    from kernelcodegen_amd import ops
    q = torch.randn(1, 8, 100, 64, device="cuda").abs()
    k, v = torch.randn(1, 8, 100, 64, device="cuda"), torch.randn(1, 8, 100, 64, device="cuda")
    k[:, :, 5] = -1e38
    k[:, :, 64:96] = -1e38                                  # a whole tile of keys whose scores overflow to -inf
    q[0, 0, 7, 3] = float("nan")
    got = ops.fmha(q, k, v, WAVEK=4)
    keep = [i for i in range(100) if i != 5 and not 64 <= i < 96]
    want = _reference(q, k[:, :, keep], v[:, :, keep], False, 64 ** -0.5)
    assert torch.isnan(got[0, 0, 7]).all() and not torch.isnan(got[0, 0, :7]).any() and not torch.isnan(got[:, 1:]).any()
    ok = ~torch.isnan(want)
    assert float((got.double() - want)[ok].norm() / want[ok].norm()) < 4e-6
    k[0, 0, 9] = float("inf")
    assert torch.isnan(ops.fmha(q, k, v, WAVEK=4)[0, 0]).all() and torch.isnan(ops.fmha(q, k, v, D2L=0)[0, 0]).all()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("form", [dict(WAVEK=4), dict()])
def test_scores_leave_the_fp32_range_only_where_they_do_scaled(form, dtype):
    """Products of queries and keys around 2^129, scaled back to 16 and at most 100; the kernels of whole tiles take them too.  A score of 100
    is off by up to three roundings to 24 bits, 2e-5 of a probability in fp32; 16 bits as above (the walk rounds scaled queries)."""
    from kernelcodegen_amd import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    q, k, v = (torch.randn(1, 8, 300, 64, generator=gen, device="cuda") for _ in range(3))
    q, k, v = (q * 2.0 ** 63).to(DTYPE[dtype]), (k * 2.0 ** 63).to(DTYPE[dtype]), v.to(DTYPE[dtype])
    got = ops.fmha(q, k, v, scale=2.0 ** -125, **form)
    want = _reference(q, k, v, False, 2.0 ** -125)
    assert float((got.double() - want).norm() / want.norm()) < (2e-5 if dtype == "f32" else TOL[dtype])
    assert torch.isfinite(ops.fmha(q, k, v, scale=2.0 ** -125, WAVEK=0)).all()
