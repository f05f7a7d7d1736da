"""LayerNorm where its row team changes (256, 1024 and 2048 rows; 64, 128, 256 and 512 lanes a row) and where the row's last vector is
moved back to its end (kernels/layernorm.hip): lengths one beside a vector, a wavefront's and a team's, and next rows under way.

The reference is fp64 of the same inputs.  Tolerances, of an element next to its row's largest: fp32 1e-5, sums of up to 8192 values in
trees of at most 32 + 6 + 3 additions (41 roundings of 2^-24 in the mean and in the variance each) and six more; 16 bits: half a
unit in the last place on top, at most 2^-8 (bf16) or 2^-11 (half) of the value.  GELU's slope is at most 1.13."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPE = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
TOL = {"f32": 1.2e-5, "bf16": 2.0 ** -8 + 1.2e-5, "f16": 2.0 ** -11 + 1.2e-5}


def _check(rows, n, dtype, gelu=False, **cfg):
    from kernelcodegen_amd import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows * 9 + n)
    draw = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    x = (draw(rows, n) * 2.0 + 0.5).to(DTYPE[dtype])
    g, b = (1.0 + 0.2 * draw(n)).to(DTYPE[dtype]), (0.2 * draw(n)).to(DTYPE[dtype])
    padded = torch.full((rows * n + 64,), 7.0, device="cuda", dtype=DTYPE[dtype])
    out = padded[32:32 + rows * n].view(rows, n)
    got = ops.layernorm(x, g, b, 1, 1e-5, gelu=gelu, out=out, **cfg)
    assert bool((padded[:32] == 7.0).all()) and bool((padded[32 + rows * n:] == 7.0).all())
    d = x.double() - x.double().mean(1, keepdim=True)
    want = d / torch.sqrt((d * d).mean(1, keepdim=True) + 1e-5) * g.double() + b.double()
    if gelu:
        want = 0.5 * want * (1.0 + torch.tanh(0.797884 * (want + 0.044715 * want ** 3)))
    err = ((got.double() - want).abs() / want.abs().amax(1, keepdim=True)).max()
    assert float(err) < TOL[dtype], (rows, n, dtype, cfg, float(err))


ROWS = [1, 7, 256, 257, 1025, 2049]
LENGTHS = [512, 513, 519, 1023, 1032, 1280, 2049, 3071, 3073, 4100, 5119, 5120, 6145, 7168, 8191, 8192]


@pytest.fixture(scope="module")
def compiled():
    """The kernels of test_lengths: one after the other they are most of its time."""
    from compile_ahead import compile_ahead
    compile_ahead([("layernorm", dict(ROWS=rows, N=n, NG=n, NB=n, EPS=1e-5, GELU=n % 2, F16=["f32", "f16", "bf16"].index(dtype)))
                   for n in LENGTHS for rows in ROWS for dtype in DTYPE])


@pytest.mark.parametrize("dtype", sorted(DTYPE))
@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("n", LENGTHS)
def test_lengths(n, rows, dtype, compiled):
    _check(rows, n, dtype, gelu=n % 2 == 1)


@pytest.mark.parametrize("rows,n,dtype", [(3200, 7777, "bf16"), (3200, 7777, "f16"), (2049, 4099, "f32"), (6500, 1281, "f32"), (3000, 8192, "f16")])
def test_held_rows(rows, n, dtype):
    _check(rows, n, dtype)


@pytest.mark.parametrize("dtype,n", [("f32", 1283), ("bf16", 1283), ("f16", 1296), ("f32", 33333), ("bf16", 12001)])
@pytest.mark.parametrize("cfg", [dict(GRID=3), dict(GRID=1000000), dict(LEAN=1, GRID=5)])
def test_forms(cfg, dtype, n):
    _check(1030, n, dtype, **cfg)


@pytest.mark.parametrize("dtype", sorted(DTYPE))
def test_empty_tail_does_not_reach_the_sums(dtype):
    """Lanes behind the row read its last vector again: infinities there must stay the row's own."""
    from kernelcodegen_amd import ops
    x = torch.zeros(300, 1281, device="cuda", dtype=DTYPE[dtype])
    x[:, ::2] = 1.0
    x[5, -1] = float("inf")
    x[9, 0] = float("nan")
    one, zero = torch.ones(1281, device="cuda", dtype=DTYPE[dtype]), torch.zeros(1281, device="cuda", dtype=DTYPE[dtype])
    y = ops.layernorm(x, one, zero, 1)
    bad = torch.zeros(300, dtype=torch.bool, device="cuda")
    bad[5] = bad[9] = True
    assert bool((torch.isnan(y).any(1) == bad).all())
