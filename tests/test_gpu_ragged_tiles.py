"""GEMM kernels on sizes that their tiles do not divide, and on fewer rows than a tile has: operands of small integers, so
that every product and sum is exact in the accumulators (|sum| <= 16 k < 2^24 for the k used here) and the comparison is
bit for bit, whatever tile and order of summation a kernel picks."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from kernelcodegen_amd import ops as _ops
    from kernelcodegen_amd._lib import lib, check
    check(lib().kcg_hip_init(0), "kcg_hip_init")
    return _ops


def _operands(m, n, k, tb, dtype, seed, batch=()):
    rs = np.random.RandomState(seed)
    a = rs.randint(-4, 5, size=batch + (m, k)).astype(np.float32)
    b = rs.randint(-4, 5, size=batch + ((n, k) if tb else (k, n))).astype(np.float32)
    want = a.astype(np.float64) @ (np.swapaxes(b, -1, -2) if tb else b).astype(np.float64)
    return torch.from_numpy(a).cuda().to(dtype), torch.from_numpy(b).cuda().to(dtype), want


def _shifted(t, elements=1):
    """The same values `elements` (one) behind a 16-byte boundary."""
    buf = torch.empty(t.numel() + elements, dtype=t.dtype, device=t.device)
    out = buf[elements:].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 != 0 and out.is_contiguous()
    return out


# tile forms of the 16-bit kernel with direct loads
FORMS = [dict(BM=256, BN=256, WM=4, WN=2), dict(BM=128, BN=128, WM=4, WN=2), dict(BM=128, BN=128, WM=4, WN=2, NBUF=3),
         dict(BM=64, BN=128, WM=2, WN=2, NBUF=3), dict(BM=64, BN=128, WM=2, WN=2, NBUF=4), dict(BM=64, BN=64, WM=2, WN=2, NBUF=4)]


@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("form", range(len(FORMS)))
def test_gemm16_every_form_at_its_edges(ops, form, tb):
    """One row or column more or less than whole tiles; a k of one tile, of a part more, of fewer tiles than buffers, of more than
    two rounds of them; odd and even counts of k-tiles, whose last iterations differ."""
    cfg = dict(FORMS[form], M16=1, D2L=1)
    bm, bn = cfg["BM"], cfg["BN"]
    ks = [64, 128, 192, 136, 200, 64 * 12, 64 * 13] if bm == 256 else [72, 136, 64 * 4, 64 * 5 + 8, 64 * 13]
    for i, (m, n) in enumerate([(bm + 1, bn + 8), (2 * bm - 1, 2 * bn - 8)]):
        for k in ks:
            a, b, want = _operands(m, n, k, tb, torch.bfloat16, 100 * form + 10 * i + k)
            out = torch.bfloat16 if i else torch.float32
            c = ops.matmul(a, b, trans_b=tb, out_dtype=out, **cfg)
            assert torch.equal(c.cpu(), torch.from_numpy(want).to(out)), (m, n, k, out)


@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 512, 512), (15, 640, 4096), (63, 520, 136), (64, 1024, 2048), (65, 584, 1000), (300, 1000, 264),
                                   (1000, 2056, 520), (257, 264, 64), (9, 64, 64), (64, 64, 72),
                                   (16, 128, 64), (16, 72, 64 * 13), (17, 136, 72), (31, 64, 320), (32, 192, 64 * 7 + 8), (33, 64, 128)])
def test_gemm16_default_forms(ops, m, n, k, tb):
    dtype = torch.float16 if (m + n) % 3 == 0 else torch.bfloat16
    out = dtype if k % 3 == 0 else torch.float32
    a, b, want = _operands(m, n, k, tb, dtype, m + n + k)
    assert torch.equal(ops.matmul(a, b, trans_b=tb, out_dtype=out).cpu(), torch.from_numpy(want).to(out))
    if m > 64:
        return
    # operands off the 16-byte boundary are taken as well, and give the same numbers
    for x, w in ((_shifted(a), b), (a, _shifted(b))):
        assert torch.equal(ops.matmul(x, w, trans_b=tb).double().cpu(), torch.from_numpy(want))


@pytest.mark.parametrize("tb", [False, True])
def test_whole_tiles_off_a_16_byte_boundary(ops, tb):
    """Operands on a multiple of four bytes keep the direct loads of whole tiles, others go through registers: the same numbers."""
    for dtype, tile in ((torch.float32, 128), (torch.bfloat16, 512), (torch.float8_e4m3fn, 512)):
        a, b, want = _operands(tile, 512, 256, tb, dtype, tile)
        run = ops.matmul if dtype != torch.float8_e4m3fn else lambda x, w, **kw: ops.matmul_fp8(x, w, 1.0, 1.0, **kw)
        cfg = {} if dtype == torch.float32 else dict(BM=256, BN=256, WM=4, WN=2)
        step = max(1, 4 // a.element_size())
        for x, w in ((_shifted(a, step), b), (a, _shifted(b, 3 * step)), (_shifted(a, 2 * step), _shifted(b, step)), (_shifted(a), _shifted(b))):
            assert torch.equal(run(x, w, trans_b=tb, **cfg).double().cpu(), torch.from_numpy(want))
    a, b, want = _operands(128, 192, 256, False, torch.float32, 3)
    cfg = dict(BM=64, BN=64, BK=32, WM=2, WN=2, WK=2, NBUF=3)
    assert torch.equal(ops.matmul(_shifted(a), _shifted(b, 2), **cfg).double().cpu(), torch.from_numpy(want))


def test_gemm16_column_count_no_multiple_of_eight(ops):
    for (m, n, k) in [(70, 515, 512), (5, 77, 128), (129, 257, 192)]:
        a, b, want = _operands(m, n, k, True, torch.bfloat16, n)
        for out in (torch.float32, torch.bfloat16):
            assert torch.equal(ops.matmul(a, b, trans_b=True, out_dtype=out).cpu(), torch.from_numpy(want).to(out))


def test_gemm16_batched(ops):
    for tb in (False, True):
        for (m, n, k) in [(65, 136, 200), (128, 64, 64), (17, 136, 200)]:
            a, b, want = _operands(m, n, k, tb, torch.float16, m, batch=(3,))
            assert torch.equal(ops.batched_matmul(a, b, trans_b=tb).double().cpu(), torch.from_numpy(want))


@pytest.mark.parametrize("tb", [False, True])
def test_gemm16_infinities_stay_in_their_rows_and_columns(ops, tb):
    """The last k-tile is moved back over values that were multiplied already, the last tiles over rows and columns that
    other tiles own: an infinity there reaches its own row and column only, and gives no NaN."""
    m, n, k = 70, 136, 200
    a, b, _ = _operands(m, n, k, tb, torch.bfloat16, 5)
    a, b = a.abs() + 1, b.abs() + 1
    a[3, 150], a[69, 0] = float("inf"), float("inf")
    b[(7, 140) if tb else (140, 7)] = float("inf")
    want = a.double().cpu() @ (b.t() if tb else b).double().cpu()
    assert not torch.isnan(want).any()
    assert torch.equal(ops.matmul(a, b, trans_b=tb).double().cpu(), want)


@pytest.mark.parametrize("tb", [True, False])
@pytest.mark.parametrize("m,n,k", [(257, 272, 128), (511, 528, 384), (300, 5008, 256), (1000, 4112, 1040), (16, 512, 512), (1, 528, 2048),
                                   (65, 80, 144), (130, 1040, 400), (700, 2064, 272), (64, 64, 128), (1100, 4112, 256)])
def test_gemm_fp8_default_forms(ops, m, n, k, tb):
    """Moved-back 256 x 256 tiles, the ring of LDS buffers (weights contiguous along k) and guarded loads of whole chunks;
    products up to 16 and |sum| <= 16 k < 2^16 stay exact in every MFMA's accumulator."""
    a, b, want = _operands(m, n, k, tb, torch.float8_e4m3fn, m + n + k)
    out = torch.float32 if m % 2 else torch.bfloat16
    assert torch.equal(ops.matmul_fp8(a, b, 0.5, 2.0, trans_b=tb, out_dtype=out).cpu(), torch.from_numpy(want).to(out))
    if m > 100:
        return
    for x, w in ((_shifted(a), b), (a, _shifted(b))):
        assert torch.equal(ops.matmul_fp8(x, w, 1.0, 1.0, trans_b=tb).double().cpu(), torch.from_numpy(want))


@pytest.mark.parametrize("ta,tb", [(True, False), (True, True)])
def test_gemm_fp8_chunks_of_a_column_major_operand(ops, ta, tb):
    m, n, k = 80, 96, 208
    a, b, want = _operands(m, n, k, tb, torch.float8_e4m3fn, 9)
    at = a.view(torch.uint8).t().contiguous().view(torch.float8_e4m3fn)
    assert torch.equal(ops.matmul_fp8(at, b, 1.0, 1.0, trans_a=ta, trans_b=tb).double().cpu(), torch.from_numpy(want))


def test_gemm_fp8_large_tiles_moved_back(ops):
    for tb in (True, False):
        for (m, n, k) in [(4001, 4128, 128), (2000, 5008, 256)]:
            a, b, want = _operands(m, n, k, tb, torch.float8_e4m3fn, m)
            c = ops.matmul_fp8(a, b, 1.0, 1.0, trans_b=tb, out_dtype=torch.float32)
            assert torch.equal(c.double().cpu(), torch.from_numpy(want))


@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("m,n,k", [(64, 64, 16), (65, 68, 20), (777, 1000, 500), (300, 460, 96), (129, 252, 1028), (64, 64, 32), (127, 64, 100),
                                   (128, 192, 64), (2000, 2000, 48), (1024, 1024, 96), (65, 67, 33), (200, 301, 99), (130, 64, 15), (257, 255, 17),
                                   (63, 64, 64), (1, 4, 4)])
def test_gemm_f32_default_forms(ops, m, n, k, tb):
    """Direct loads with moved-back tiles and k-tiles (rows of whole 16-byte chunks), 16-byte loads at any row length with
    the last k-tile guarded, and the guarded form where an operand holds no whole tile."""
    a, b, want = _operands(m, n, k, tb, torch.float32, m + n + k)
    assert torch.equal(ops.matmul(a, b, trans_b=tb).double().cpu(), torch.from_numpy(want))
    for x, w in ((_shifted(a), b), (a, _shifted(b))):
        assert torch.equal(ops.matmul(x, w, trans_b=tb).double().cpu(), torch.from_numpy(want))


F32_FORMS = [dict(BM=256, BN=256, BK=16, WM=4, WN=4), dict(BM=128, BN=128, BK=16, WM=4, WN=4), dict(BM=64, BN=64, BK=16, WM=2, WN=2),
             dict(BM=64, BN=64, BK=32, WM=2, WN=2), dict(BM=64, BN=64, BK=32, WM=2, WN=2, WK=2, NBUF=3), dict(BM=64, BN=64, BK=32, WM=2, WN=2, NBUF=4)]


@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("form", range(len(F32_FORMS)))
def test_gemm_f32_direct_load_forms_at_their_edges(ops, form, tb):
    cfg = F32_FORMS[form]
    bm, bk = cfg["BM"], cfg["BK"]
    for i, (m, n) in enumerate([(bm + 1, bm + 4), (2 * bm - 1, 2 * bm - 4)]):
        for k in (bk, bk + 4, 3 * bk - 4, 5 * bk - 4, 9 * bk):      # (one and two k-tiles, fewer than there are buffers, too)
            a, b, want = _operands(m, n, k, tb, torch.float32, 100 * form + 10 * i + k, batch=(2,))
            assert torch.equal(ops.batched_matmul(a, b, trans_b=tb, **cfg).double().cpu(), torch.from_numpy(want)), (m, n, k)


@pytest.mark.parametrize("ta,tb", [(True, False), (True, True)])
def test_gemm_f32_column_major_left_operand(ops, ta, tb):
    for (m, n, k) in [(70, 75, 33), (131, 129, 50), (64, 200, 19)]:
        a, b, want = _operands(m, n, k, tb, torch.float32, m)
        assert torch.equal(ops.matmul(a.t().contiguous(), b, trans_a=True, trans_b=tb).double().cpu(), torch.from_numpy(want))


@pytest.mark.parametrize("tb", [False, True])
def test_gemm_f32_infinities_stay_in_their_rows_and_columns(ops, tb):
    for (m, n, k) in [(70, 136, 100), (70, 135, 101)]:
        a, b, _ = _operands(m, n, k, tb, torch.float32, 5)
        a, b = a.abs() + 1, b.abs() + 1
        a[3, 90], a[69, 0] = float("inf"), float("inf")
        b[(7, 85) if tb else (85, 7)] = float("inf")
        want = a.double().cpu() @ (b.t() if tb else b).double().cpu()
        assert not torch.isnan(want).any()
        assert torch.equal(ops.matmul(a, b, trans_b=tb).double().cpu(), want)


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-6), (torch.float16, 2 ** -10), (torch.bfloat16, 2 ** -7)])
@pytest.mark.parametrize("rows,n", [(3, 259), (9, 1001), (2, 32767), (3, 256), (4, 255), (1200, 1003), (4200, 257), (600, 2050), (600, 8192),
                                    (300, 4100), (40, 31999)])
def test_rows_of_any_length(ops, rows, n, dtype, tol):
    """Softmax and LayerNorm over rows that start anywhere: results within one rounding of the type (2^-10 and 2^-7: one ulp
    above 1, relative; fp32 sums of n <= 2^15 terms in trees stay below 1e-6), and nothing written behind the result."""
    gen = torch.Generator(device="cuda").manual_seed(rows * n)
    x = torch.randn((rows, n), generator=gen, device="cuda").to(dtype)
    g = (torch.rand((n,), generator=gen, device="cuda") + 0.5).to(dtype)
    b = torch.randn((n,), generator=gen, device="cuda").to(dtype)
    x64 = x.double()
    want = torch.softmax(x64, -1)
    y = ops.softmax(x)
    assert ((y.double() - want).abs() <= tol * want + (2.0 ** -24 if dtype == torch.float16 else 0.0)).all()
    z = x.clone()
    assert torch.equal(ops.softmax(z, inplace=True), y)
    c = x64 - x64.mean(-1, keepdim=True)
    want = c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-5) * g.double() + b.double()
    for out in (None, torch.full((rows + 1, n), 7.0, device="cuda", dtype=dtype)):
        got = ops.layernorm(x, g, b, -1, out=None if out is None else out[:rows])
        assert ((got.double() - want).norm() <= tol * want.norm()).all()
        assert out is None or (out[rows:] == 7.0).all()


def test_softmax_rows_of_infinities_and_nan(ops):
    x = torch.randn((4, 1001), device="cuda")
    x[0, 500:] = float("-inf")
    x[1, 1000] = float("nan")
    x[2, :1000] = float("-inf")
    y, want = ops.softmax(x), torch.softmax(x.double(), -1)
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    assert ((y.double() - want).abs()[[0, 2, 3]] <= 1e-6).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 1e-2), (torch.float16, 2e-3), (torch.float32, 4e-6)])
@pytest.mark.parametrize("b,h,s,d", [(1, 8, 333, 64), (1, 3, 64, 64), (1, 3, 65, 128), (1, 5, 256, 128), (1, 32, 1100, 128), (2, 64, 512, 128),
                                     (1, 80, 448, 128), (1, 90, 384, 128), (1, 64, 600, 128), (1, 80, 768, 128)])
def test_attention_on_small_launches(ops, b, h, s, d, dtype, tol, causal):
    """128 queries per workgroup and no pairs of query tiles where the launch leaves compute units empty, 64 for fp32 under
    the mask; the tolerances are those of the other attention tests (16-bit probabilities, fp32 sums)."""
    gen = torch.Generator(device="cuda").manual_seed(s + d)
    q, k, v = (torch.randn((b, h, s, d), generator=gen, device="cuda").to(dtype) for _ in range(3))
    got = ops.fmha(q, k, v, causal=causal).double()
    for i in range(b):
        scores = (q[i].double() @ k[i].double().transpose(-1, -2).contiguous()) * d ** -0.5
        if causal:
            scores.masked_fill_(torch.ones((s, s), dtype=torch.bool, device="cuda").triu(1), float("-inf"))
        want = torch.softmax(scores, -1) @ v[i].double()
        assert ((got[i] - want).norm() <= tol * want.norm()).item()
