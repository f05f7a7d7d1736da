"""When a product takes the form whose wavefronts split k, and that every form compiles into registers (no GPU needed)."""
import pytest

from kernelcodegen_amd import _lib, runtime as R
from test_gemm_forms import scratch_bytes


def text_of(family, **params):
    return R.emit_kernel(family, "kernel0", **R.launch_params(family, params))[0]


SPLIT = "#define GW_WK"


def test_only_aligned_products_without_wishes_split_k():
    """Launched from here, on operands known to be aligned, in rows of whole chunks, A contiguous along k; all else keeps its kernel."""
    small = dict(M=8, N=1024, K=4096, TB=1, ALIGN=16)
    assert SPLIT in text_of("gemm_bf16", **small) and SPLIT in text_of("gemm_fp8", **small)
    assert SPLIT not in R.emit_kernel("gemm_bf16", "kernel0", **small)[0]
    for other in (dict(ALIGN=0), dict(K=4097), dict(K=4100), dict(TB=0, N=1020), dict(M=4096, N=4096), dict(BM=64, BN=64), dict(D2L=0), dict(WAVEK=0), dict(TA=1)):
        assert SPLIT not in text_of("gemm_bf16", **dict(small, **other)), other
    for other in (dict(ALIGN=0), dict(K=4104), dict(N=1032, TB=0), dict(SCALE_PTR=1), dict(BM=64, BN=64), dict(WAVEK=0)):
        assert SPLIT not in text_of("gemm_fp8", **dict(small, **other)), other
    single = dict(M=256, N=256, K=1024, ALIGN=16)
    for same in (dict(), dict(TB=1), dict(K=1023), dict(N=255), dict(BATCH=3)):
        assert SPLIT in text_of("gemm_f32", **dict(single, **same)), same
    for other in (dict(ALIGN=0), dict(M=4096, N=4096), dict(M=60), dict(TA=1), dict(WK=2), dict(D2L=0), dict(WAVEK=0)):
        assert SPLIT not in text_of("gemm_f32", **dict(single, **other)), other


@pytest.mark.parametrize("bad", [dict(WAVEK=17), dict(TM=9), dict(TN=17), dict(DEPTH=17), dict(WAVEK=16, K=64), dict(TM=8, TN=8, WAVEK=8), dict(TB=0, VW=16),
                                 dict(TB=0, TN=2, VW=4), dict(ALIGN=0), dict(K=1001), dict(TA=1)])
def test_what_is_asked_for_and_does_not_fit_is_refused(bad):
    with pytest.raises(_lib.KcgError):
        R.emit_kernel("gemm_bf16", "kernel0", **dict(dict(M=100, N=512, K=1024, TB=1, ALIGN=16, WAVEK=4), **bad))


@pytest.mark.parametrize("family,extra", [("gemm_bf16", dict(OUT_BF16=1)), ("gemm_bf16", dict(F16=1, RELU=1)), ("gemm_fp8", dict(OUT_BF16=1)), ("gemm_f32", dict())])
@pytest.mark.parametrize("tb", [0, 1])
def test_every_chosen_form_stays_in_registers(family, extra, tb):
    seen = set()
    for m, n, k in [(1, 512, 528), (8, 1024, 4096), (16, 4096, 4096), (64, 1024, 4096), (100, 1024, 4096), (200, 1024, 4096), (300, 640, 1216), (256, 256, 2048),
                    (300, 300, 1002), (500, 500, 500), (914, 752, 1227)]:
        if family != "gemm_f32" and (k % 16 or n % 16):
            continue
        text = text_of(family, M=m, N=n, K=k, TB=tb, ALIGN=16, **extra)
        if SPLIT in text:
            form = tuple(l.split()[2] for l in text.splitlines() if l.startswith(("#define GW_TM", "#define GW_TN", "#define GW_WK", "#define GW_DEPTH")))
            if form not in seen:
                seen.add(form)
                assert scratch_bytes(R.compile_to_code(R.prelude() + text)) == 0, (m, n, k, form)
    assert len(seen) >= 3, seen


WISHES = {"gemm_bf16": dict(BM=64, BN=64, BK=64, WM=2, WN=2, GROUP_M=4, M16=1, D2L=1, BTR=0, BPAD=0, STAGES=1, NBUF=2, SK_UNITS=0, INTERLEAVE=1, SETPRIO=1,
                            STAGE_C=0, KROT=1, STAGGER=1, M16_DEAL=1),
          "gemm_fp8": dict(BM=64, BN=64, BK=128, WM=2, WN=2, GROUP_M=4, D2L=0, BTR=1, STAGES=1, PREFETCH=1, ROTATE=1, PINGPONG=1, PERSIST=0, STAGE_C=0, NT_STORE=1, STAGGER=1),
          "gemm_f32": dict(BM=64, BN=64, BK=32, WM=2, WN=2, WK=1, NBUF=2, PAD=4, GROUP_M=4, D2L=1)}


@pytest.mark.parametrize("family,key", [(f, k) for f in sorted(WISHES) for k in sorted(WISHES[f])])
def test_a_wish_that_the_split_has_no_use_for_is_not_dropped(family, key):
    """Each parameter of the kernels of whole tiles, by itself, keeps the product on them."""
    small = dict(M=64, N=256, K=1024, TB=1, ALIGN=16)
    assert SPLIT in text_of(family, **small)
    try:
        assert SPLIT not in text_of(family, **dict(small, **{key: WISHES[family][key]}))
    except _lib.KcgError:
        pass                              # (refused as it would be without the split)


@pytest.mark.parametrize("family,problem", [("gemm_bf16", dict(M=64, N=256, K=1024, TB=1, ALIGN=16)), ("gemm_f32", dict(M=256, N=256, K=1024, ALIGN=16)),
                                            ("gemm_fp8", dict(M=64, N=256, K=1024, TB=1, ALIGN=16)), ("fmha_bf16", dict(B=1, H=8, S=333, D=64)), ("fmha_f32", dict(B=1, H=8, S=333, D=64))])
def test_without_the_split_a_launch_has_the_forms_of_whole_tiles(family, problem):
    assert text_of(family, WAVEK=0, **problem) == R.emit_kernel(family, "kernel0", FILL=1, **problem)[0] != text_of(family, **problem)


@pytest.mark.parametrize("family,tb,sizes", [("gemm_fp8", 0, [(40, 4800, 3968), (33, 3840, 2816), (40, 5776, 3888), (37, 4096, 3072), (63, 7072, 3712), (545, 544, 4032)]),
                                             ("gemm_f32", 1, [(664, 1111, 3520), (320, 901, 3205, 2), (1420, 475, 3560), (244, 174, 4052, 15)])])
def test_products_of_the_largest_tiles_stay_in_registers(family, tb, sizes):
    """Products for which eight wavefronts on the largest tiles, two steps in flight, would be the form of least modelled time."""
    for m, n, k, *batch in sizes:
        text = text_of(family, M=m, N=n, K=k, TB=tb, ALIGN=16, BATCH=batch[0] if batch else 1)
        assert scratch_bytes(R.compile_to_code(R.prelude() + text)) == 0, (m, n, k, batch)


@pytest.mark.parametrize("k,tb", [(1001, 1), (1002, 0), (1024, 1)])
def test_loads_declare_the_alignment_that_rows_have(k, tb, tmp_path):
    """fp32 rows of no whole 16-byte chunks start on any multiple of four bytes: no load of the operands may promise more."""
    import re
    import subprocess
    from kernelcodegen_amd import build as B
    src, out = tmp_path / "k.hip", tmp_path / "k.ll"
    src.write_text(R.prelude() + text_of("gemm_f32", M=256, N=256, K=k, TB=tb, ALIGN=16, WAVEK=4, TM=2, TN=2, **({} if tb else dict(VW=1))))
    subprocess.run([B.HIPCC] + B.DEVICE_FLAGS + ["--cuda-device-only", "-S", "-emit-llvm", str(src), "-o", str(out)], check=True, stderr=subprocess.PIPE)
    aligned = {int(a) for a in re.findall(r"load <4 x i32>, ptr addrspace\(1\) [^\n]*?, align (\d+)", out.read_text())}
    assert aligned == ({16} if k % 4 == 0 else {4}), aligned
