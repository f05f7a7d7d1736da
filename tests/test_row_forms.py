"""The forms that LayerNorm and softmax kernels get for a row length, seen in the emitted parameters and the compiled code (no GPU
needed)."""
import os
import re
import subprocess

import pytest

from kernelcodegen_amd import runtime as R
from test_gemm_forms import defines, scratch_bytes

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
TYPES = {"f32": 0, "f16": 1, "bf16": 2}


def code_object(family, **params):
    text, _ = R.emit_kernel(family, "kernel0", **params)
    return R.compile_to_code(R.prelude() + text)


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
@pytest.mark.parametrize("n,vw", [(320, 4), (448, 4), (768, 8), (1000, 8), (2048, 8), (5120, 8)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_whole_rows_of_softmax_are_loaded_as_vectors_only(tmp_path, dtype, n, vw):
    """A row length that the vector width divides needs no load of single elements, also where the last vectors of the team
    lie behind the row."""
    path = tmp_path / "kernel.hsaco"
    path.write_bytes(code_object("softmax", ROWS=1255, N=n, INPLACE=0, F16=TYPES[dtype], VW=vw))
    listing = subprocess.run([OBJDUMP, "-d", str(path)], capture_output=True, text=True, check=True).stdout
    loads = set(re.findall(r"global_load_\w+", listing))
    assert loads == {"global_load_dwordx%d" % (vw // 2)}, loads


@pytest.mark.parametrize("dtype", sorted(TYPES))
@pytest.mark.parametrize("n", [1001, 4096, 8191, 8192, 12001, 16381, 16384, 20001, 24576, 24584, 26565, 28135, 28136, 32001, 32768])
def test_layernorm_keeps_its_rows_in_registers(n, dtype):
    """Row, prefetched row, gamma and beta: whatever does not fit a lane's registers is read again, not kept in scratch memory (32
    bytes: a few addresses)."""
    for gelu in (0, 1):
        scratch = scratch_bytes(code_object("layernorm", ROWS=2000, N=n, NG=n, NB=n, EPS=1e-5, GELU=gelu, F16=TYPES[dtype]))
        assert scratch <= 32, (n, dtype, scratch)


def lanes_in_fours(n, most):
    """Lanes that share a row when each takes four vectors of four."""
    lanes = 64
    while lanes * 16 < n and lanes < most:
        lanes *= 2
    return lanes


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rows", [1, 64, 300, 1000])
def test_layernorm_of_16_bit_rows_keeps_its_lanes_and_its_alignment(rows, dtype):
    """Wider vectors take fewer loads of each lane and not fewer lanes: a small launch lasts as long as a lane's chain.  Rows that
    fours divide and eights do not stay aligned in fours; 768 elements fill a wavefront in fours only."""
    def form(n):
        return defines("layernorm", ROWS=rows, N=n, NG=n, NB=n, EPS=1e-5, F16=TYPES[dtype])
    for n in (1024, 2048, 3000, 3072, 4096, 5120, 8192):
        d = form(n)
        assert d["LN_VW"] == "8" and int(d["LN_TPR"]) >= lanes_in_fours(n, 512), n
    for n in (1028, 1500, 2044, 3892, 5004, 7004):
        d = form(n)
        assert d["LN_VW"] == "4" and int(d["LN_TPR"]) == lanes_in_fours(n, 512), n
    assert form(768)["LN_VW"] == "4" and form(1000)["LN_VW"] == "8"
    for n in (2503, 3893):          # single elements while every row has a workgroup of its own, then eights on as many lanes
        d = form(n)
        assert d["LN_VW"] == ("8" if rows > 512 else "1") and (rows <= 512 or int(d["LN_TPR"]) == lanes_in_fours(n, 512)), n


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("rows", [1, 64, 500])
def test_softmax_of_16_bit_rows_keeps_its_lanes_and_its_alignment_on_small_launches(rows, dtype):
    def form(n, r=rows):
        return defines("softmax", ROWS=r, N=n, INPLACE=0, F16=TYPES[dtype])
    for n in (1024, 2048, 3000, 3072, 4096, 5120, 8192):
        d = form(n)
        assert d["SM_VW"] == "8" and int(d["SM_TPR"]) >= lanes_in_fours(n, 1024), n
    for n in (1028, 1500, 2044, 3892, 5004, 8188):
        d = form(n)
        assert d["SM_VW"] == "4" and int(d["SM_TPR"]) == lanes_in_fours(n, 1024), n
    assert int(form(4096, 16384)["SM_TPR"]) == 128 and form(3892, 16384)["SM_VW"] == "8" and form(1500, 4000)["SM_VW"] == "4"
    assert int(form(3893, 1000)["SM_TPR"]) == lanes_in_fours(3893, 1024) and form(3893, 1000)["SM_VW"] == "8"


@pytest.mark.parametrize("dtype", sorted(TYPES))
@pytest.mark.parametrize("rows,n", [(1 << 26, 512), (1 << 25, 1024), (1 << 24, 5000), (1 << 28, 64), ((1 << 32) - 1, 8), (5000000, 32000)])
def test_a_layernorm_of_very_many_rows_is_one_launch(rows, n, dtype):
    """Fewer than 2^32 threads, the most that a launch takes; workgroups walk the rows that are left."""
    text, info = R.emit_kernel("layernorm", "kernel0", ROWS=rows, N=n, NG=n, NB=n, EPS=1e-5, F16=TYPES[dtype])
    assert info["grid"][0] * info["block"][0] < 1 << 32
    assert "#define LN_GRID %d\n" % info["grid"][0] in text


@pytest.mark.parametrize("rows,n,grid", [(5888, 2639, 768), (8814, 1497, 768), (4714, 3318, 768), (16004, 3999, 512), (4096, 4096, 512), (16384, 4096, 512), (5151, 5435, 512), (11807, 1101, 512),
                                         (16384, 832, 768)])
def test_held_layernorm_rows_walk_on_few_workgroups(rows, n, grid):
    """fp32 rows that start off the vectors on somewhat more of them than whole ones, while they are not far beyond the caches."""
    _, info = R.emit_kernel("layernorm", "kernel0", ROWS=rows, N=n, NG=n, NB=n, EPS=1e-5)
    assert info["grid"][0] == grid


@pytest.mark.parametrize("rows,n,ng,branches", [(138, 387, 387, 0), (13, 2723, 1, 0), (2, 3989, 1, 0), (445, 10115, 10115, 1), (12087, 8743, 8743, 1), (16384, 387, 387, 1), (4096, 1024, 1024, 0)])
def test_layernorm_loads_behind_branches_where_they_are_faster(rows, n, ng, branches):
    """Workgroups that walk, and rows of more than eight single elements a lane; not shorter ones with a workgroup each."""
    text, _ = R.emit_kernel("layernorm", "kernel0", **R.launch_params("layernorm", dict(ROWS=rows, N=n, NG=ng, NB=ng, EPS=1e-5, F16=1)))
    lines = [l for l in text.splitlines() if l.startswith("#define LN_")]
    done = subprocess.run(["g++", "-E", "-P", "-x", "c", "-"], input="\n".join(lines) + "\n#if LN_APART\nbranches 1\n#else\nbranches 0\n#endif\n", capture_output=True, text=True, check=True)
    assert done.stdout.split()[-2:] == ["branches", str(branches)]
