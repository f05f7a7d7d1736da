"""Which form of the GEMM kernels a set of parameters gets, and that every set the emitter accepts compiles (no GPU needed)."""
import pytest

from kernelcodegen_amd import _lib, runtime as R

TILE256 = dict(BM=256, BN=256, WM=4, WN=2)
TILE128 = dict(BM=128, BN=128, WM=4, WN=2)


def defines(family, **params):
    """The parameters in front of the emitted kernel (its leading #define lines) as a dict."""
    text, _ = R.emit_kernel(family, "kernel0", **params)
    out = {}
    for line in text.splitlines():
        if not line.startswith("#define "):
            break
        out.update([line.split(None, 2)[1:]])
    return out


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("tile", [TILE256, TILE128])
@pytest.mark.parametrize("extra", [dict(OUT_BF16=1), dict(STAGE_C=1), dict(OUT_BF16=1, D2L=1), dict(K=520)])
def test_rows_are_clamped_in_tiles_of_at_most_64_rows_only(tile, tb, extra):
    """A 256-row tile leaves through LDS as whole rows, those past the last included: fewer rows than such a tile must not
    reach the 16x16x32 form (its stores would run past the end of C)."""
    params = dict(dict(M=100, N=512, K=512, TB=tb, ALIGN=16, **tile), **extra)
    with pytest.raises(_lib.KcgError):
        R.emit_kernel("gemm_bf16", "kernel0", M16=1, **params)
    params.pop("D2L", None)
    d = defines("gemm_bf16", **params)
    assert d["GB_EDGE"] == "1" and "GB_CLAMP" not in d and "GB_SHIFT" not in d and "GB_STAGE_C" not in d


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("m,n,k", [(300, 512, 520), (100, 512, 512), (40, 512, 512), (300, 520, 576), (256, 512, 520), (300, 512, 512)])
@pytest.mark.parametrize("tile", [TILE128, TILE256, dict(BM=64, BN=64, WM=2, WN=2), dict(BM=64, BN=128, WM=2, WN=2), dict(BM=128, BN=256, WM=2, WN=4)])
def test_tiles_asked_for_without_direct_loads_are_refused_or_compile(tile, m, n, k, tb):
    """M16 without D2L: row-major weights in tiles of fewer than 256 columns go through registers then, which can move tiles
    back but neither a k-tile nor clamp rows; the emitter says so, or what it emits compiles."""
    for extra in (dict(), dict(D2L=0)):
        params = dict(M=m, N=n, K=k, TB=tb, ALIGN=16, M16=1, **dict(tile, **extra))
        try:
            text, _ = R.emit_kernel("gemm_bf16", "kernel0", **params)
        except _lib.KcgError:
            continue
        d = defines("gemm_bf16", **params)
        if "GB_D2L" not in d:
            assert "GB_KTAIL" not in d and "GB_CLAMP" not in d, params
        if m + k < 900 and n == 512:          # every branch above with few kernels to compile
            assert R.compile_to_code(R.prelude() + text)


def scratch_bytes(code):
    """Private segment size in a code object's metadata (one kernel): scratch memory per lane."""
    at = code.index(b".private_segment_fixed_size") + len(b".private_segment_fixed_size")
    size = {0xcc: 1, 0xcd: 2, 0xce: 4}.get(code[at], 0)          # MessagePack: uint8, uint16, uint32, else the number itself
    return int.from_bytes(code[at + 1:at + 1 + size], "big") if size else code[at]


# a size for each form of the 16-bit kernel that is chosen by itself: 256 x 256 tiles whole and moved back, 128 x 128 with two
# and three buffers, 64 x 128 with three and four, 64 x 64, 32 x 64
SIZES = [(4096, 4096), (1000, 11008), (2048, 4096), (1000, 2048), (300, 11008), (512, 4096), (128, 4096), (16, 4096)]


@pytest.mark.parametrize("k", [64, 128, 192, 320, 384, 1088, 1152, 72, 136, 200, 584, 1040, 1104])
def test_no_form_of_the_16_bit_gemm_keeps_registers_in_scratch_memory(k):
    """Any count of k-tiles, odd or even, whole or with a moved-back last one; 32 bytes are the few address registers that a
    16-bit result's row stores cost."""
    seen = set()
    for m, n in SIZES:
        for tb, out in ((0, 1), (1, 0)):
            params = dict(M=m, N=n, K=k, TB=tb, OUT_BF16=out, ALIGN=16)
            text, _ = R.emit_kernel("gemm_bf16", "kernel0", **params)
            d = defines("gemm_bf16", **params)
            seen.add((d["GB_BM"], d["GB_BN"], d.get("GB_NBUF", "2")))
            scratch = scratch_bytes(R.compile_to_code(R.prelude() + text))
            assert d["GB_D2L"] == "1" and scratch <= 32, params
    assert {("64", "64", "4"), ("32", "64", "4")} <= seen and (k % 64 or ("256", "256", "2") in seen), seen



def test_guarded_fp8_loads_in_chunks():
    """Every aligned ragged tile but those of up to 128 x 128 of two k-contiguous operands in whole k-tiles."""
    def wide(**params):
        return defines("gemm_fp8", **dict(dict(M=700, N=816, K=512, TB=1, ALIGN=16, D2L=0, BM=128, BN=128), **params)).get("GF_WIDE")
    assert wide() is None and wide(BM=64, BN=64) is None and wide(ALIGN=0, K=528) is None
    assert wide(K=528) == "1" and wide(TB=0) == "1" and wide(BM=256, BN=256) == "1" and wide(M=704, TA=1) == "1"


@pytest.mark.parametrize("m,n,k,guarded", [(2000, 5504, 512, 1), (1000, 11008, 1024, 1), (2000, 2816, 1024, 1), (1000, 5504, 256, 1),
                                           (2000, 2816, 2048, 0), (2447, 5504, 1024, 0), (700, 5504, 512, 0), (300, 11008, 512, 0), (2447, 2816, 528, 0)])
def test_shallow_fp8_products_keep_the_guarded_tiles(m, n, k, guarded):
    """Which kernel a ragged product of two k-contiguous operands takes by its depth and by how much of the part its tiles fill."""
    d = defines("gemm_fp8", M=m, N=n, K=k, TB=1, ALIGN=16)
    assert ("GF_M" in d) == bool(guarded), d
    if guarded:
        assert d["GF_BM"] == d["GF_BN"] == "128" and "GF_WIDE" not in d
    d = defines("gemm_fp8", M=m, N=n, K=k, TB=0, ALIGN=16)
    assert d.get("G8_SHIFT", d.get("GF_WIDE")) == "1"
