"""When attention takes the form whose wavefronts split the keys, and that every form compiles into registers (no GPU needed)."""
import pytest

from kernelcodegen_amd import _lib, runtime as R
from test_gemm_forms import scratch_bytes

SPLIT = "#define FW_WK"


def text_of(family, **params):
    return R.emit_kernel(family, "kernel0", **R.launch_params(family, params))[0]


@pytest.mark.parametrize("family", ["fmha_bf16", "fmha_f32"])
def test_only_small_launches_without_wishes_split_the_keys(family):
    small = dict(B=1, H=8, S=333, D=64, SCALE=0.1, FILL=1)
    assert SPLIT in text_of(family, **small) and SPLIT in text_of(family, **dict(small, D=128, CAUSAL=1))
    # fp32 at head dim 128 in whole tiles: direct loads, which give the bits that the same kernel gives without them
    assert (SPLIT in text_of(family, **dict(small, D=128, S=512))) == (family == "fmha_bf16")
    assert SPLIT not in R.emit_kernel(family, "kernel0", **small)[0]
    for other in (dict(FILL=0), dict(B=8, H=32, S=2048), dict(D=96), dict(D=32), dict(BR=64), dict(BC=32), dict(WAVEK=0)):
        assert SPLIT not in text_of(family, **dict(small, **other)), other


@pytest.mark.parametrize("bad", [dict(WAVEK=17), dict(QB=3), dict(D=96), dict(D=256), dict(SCALE=-1.0), dict(WAVEK=16, D=128), dict(B=0)])
def test_what_is_asked_for_and_does_not_fit_is_refused(bad):
    with pytest.raises(_lib.KcgError):
        R.emit_kernel("fmha_bf16", "kernel0", **dict(dict(B=1, H=8, S=333, D=64, WAVEK=4), **bad))


@pytest.mark.parametrize("heads,s", [(1 << 23, 129), (1 << 22, 333)])
def test_a_launch_has_fewer_than_2_to_the_32_threads(heads, s):
    """Very many heads: wavefronts that walk the keys, or 64 queries a workgroup, fit one launch where splitting over 32 does not."""
    many = dict(B=1, H=heads, S=s, D=64, CAUSAL=1, SCALE=0.1)
    _, info = R.emit_kernel("fmha_bf16", "kernel0", **R.launch_params("fmha_bf16", many))
    assert info["grid"][0] * info["block"][0] < 1 << 32
    with pytest.raises(_lib.KcgError):
        R.emit_kernel("fmha_bf16", "kernel0", WAVEK=2, **many)


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("family,extra", [("fmha_bf16", dict()), ("fmha_bf16", dict(F16=1)), ("fmha_bf16", dict(OUT_BF16=0)), ("fmha_f32", dict())])
def test_every_chosen_form_stays_in_registers(family, extra, causal):
    seen = set()
    for heads in (8, 32, 64):
        for s in (33, 64, 100, 333, 777, 2048):
            for d in (64, 128):
                text = text_of(family, B=1, H=heads, S=s, D=d, CAUSAL=causal, SCALE=0.1, FILL=1, **extra)
                if SPLIT in text:
                    form = (d, s % 32 == 0) + tuple(l.split()[2] for l in text.splitlines() if l.startswith(("#define FW_WK", "#define FW_QB", "#define FW_EU")))
                    if form not in seen:
                        seen.add(form)
                        assert scratch_bytes(R.compile_to_code(R.prelude() + text)) == 0, (heads, s, form)
    assert len(seen) >= 5, seen


@pytest.mark.parametrize("scale", [64 ** -0.5, 1.0, 3.0, 2.0 ** -125, 2.0 ** -130, 1e30])
@pytest.mark.parametrize("family,f16", [("fmha_f32", 0), ("fmha_bf16", 0), ("fmha_bf16", 1)])
def test_queries_are_scaled_by_a_power_of_two(family, f16, scale):
    """2^FW_QEXP, a normal number of at most 1, times FW_C is the scale; IEEE half, whose products stay in the fp32 range, is left alone."""
    text = text_of(family, B=1, H=8, S=333, D=64, SCALE=scale, F16=f16, WAVEK=4)
    define = {l.split()[1]: l.split()[2] for l in text.splitlines() if l.startswith(("#define FW_QEXP", "#define FW_C "))}
    c, down = float.fromhex(define["FW_C"].rstrip("f")), int(define["FW_QEXP"])
    want = scale * 1.4426950408889634
    assert abs(c * 2.0 ** down / want - 1) < 2.0 ** -24 or (f16 and scale < 2.0 ** -126)
    assert down == 0 if f16 or want >= 1 else (-126 <= down < 0 and (1 <= c < 2 or down == -126))


@pytest.mark.parametrize("family,wish", [("fmha_bf16", dict(VPAD=48)), ("fmha_bf16", dict(QW=1)), ("fmha_bf16", dict(OCC=1)), ("fmha_bf16", dict(STAGE_O=0)), ("fmha_bf16", dict(PERSIST=0)),
                                         ("fmha_bf16", dict(PAIR=0)), ("fmha_bf16", dict(D2L=0)), ("fmha_f32", dict(OCC=1)), ("fmha_f32", dict(PAIR=0)), ("fmha_f32", dict(D2L=0))])
def test_a_wish_that_the_split_has_no_use_for_is_not_dropped(family, wish):
    assert SPLIT not in text_of(family, B=1, H=8, S=333, D=64, SCALE=0.1, **wish)


@pytest.mark.parametrize("family,heads,s,d,split", [("fmha_bf16", 183, 362, 64, False), ("fmha_bf16", 371, 1126, 64, False), ("fmha_bf16", 234, 400, 64, False), ("fmha_bf16", 291, 270, 64, True),
                                                    ("fmha_bf16", 8, 333, 64, True), ("fmha_f32", 255, 91, 128, False), ("fmha_f32", 225, 89, 128, False), ("fmha_f32", 97, 970, 64, True)])
def test_more_workgroups_than_the_part_holds_rarely_split(family, heads, s, d, split):
    """Under the mask, launches that were measured slower split than walked beside such as were faster."""
    assert (SPLIT in text_of(family, B=1, H=heads, S=s, D=d, CAUSAL=1, SCALE=0.1)) == split
