"""What a bound launch passes on, and what the operators' keys keep apart, without a GPU: the entry points that would launch are
replaced by recorders."""
import ctypes as C
import struct

import pytest

torch = pytest.importorskip("torch")

from kernelcodegen_amd import ops, runtime as R


class Recorder:
    """Stands for the library: keeps what kcg_hip_launch_packed was given."""

    def __init__(self):
        self.calls = []

    def kcg_hip_launch_packed(self, handle, dims, stream, slots, n):
        self.calls.append((list((C.c_uint32 * 7).from_address(dims)), stream, bytes(slots), n))
        return 0


@pytest.fixture
def recorder(monkeypatch):
    r = Recorder()
    monkeypatch.setattr(R, "lib", lambda: r)
    monkeypatch.setattr(R, "_current_stream", lambda: lambda: 77)
    return r


def test_scalars_beyond_fp32_become_infinity(recorder):
    """As a C float argument: a finite number above the fp32 range is not an error."""
    kern = R.Kernel(None, 5, dict(grid=(1, 2, 3), block=(64, 1, 1), lds_bytes=9, num_args=5, workspace_bytes=0))
    run = kern.bind(scalars=2)
    for value in (0.5, -2.0, 1e39, -1e39, 3.4028235677973366e38, 1e-46, float("inf"), float("-inf"), 0.1, float("nan")):
        run(1, 2, 3, value, 0.25)
        dims, stream, slots, n = recorder.calls[-1]
        assert dims == [1, 2, 3, 64, 1, 1, 9] and stream == 77 and n == 5
        assert slots[:24] == struct.pack("<3Q", 1, 2, 3)
        assert slots[24:28] == bytes(C.c_float(value)) and slots[32:36] == bytes(C.c_float(0.25))


@pytest.fixture
def kernels(monkeypatch):
    """The parameters that the operators ask kernels for; every kernel's bound launch does nothing."""
    asked = []

    class Kern:
        info = dict(workspace_bytes=0)

        def bind(self, scalars=0):
            return lambda *values: None

    def get_kernel(family, **params):
        asked.append((family, params))
        return Kern()

    monkeypatch.setattr(R, "get_kernel", get_kernel)
    monkeypatch.setattr(ops, "_need_cuda", lambda *ts: None)
    monkeypatch.setattr(ops, "_bound", {})
    return asked


def test_parameters_that_follow_from_the_operands_cannot_be_overridden(kernels):
    """The result's tensor is allocated from out_dtype and the operands: a kernel told otherwise would write another size."""
    a, b = torch.zeros(64, 64, dtype=torch.float16), torch.zeros(64, 64, dtype=torch.float16)
    for key in ("OUT_BF16", "F16", "M", "N", "K", "BATCH", "TA", "TB"):
        with pytest.raises(TypeError):
            ops.batched_matmul(a, b, **{key: 1})
    f8 = a.to(torch.float8_e4m3fn)
    with pytest.raises(TypeError):
        ops.matmul_fp8(f8, f8, 1.0, 1.0, OUT_BF16=1)
    assert not kernels
    ops.batched_matmul(a, b, ALIGN=0, D2L=0)
    assert kernels[0][1]["ALIGN"] == 0 and kernels[0][1]["D2L"] == 0


def test_an_axis_is_a_whole_number_on_every_call(kernels):
    """1.0 == 1 as a dictionary key: a call that is refused must not find the launch that an accepted one has bound."""
    x, g = torch.zeros(4, 8), torch.zeros(8)
    ops.layernorm(x, g, g, 1)
    with pytest.raises(TypeError):
        ops.layernorm(x, g, g, 1.0)
    ids = torch.zeros(3, dtype=torch.int64)
    ops.gather(x, ids, 1)
    with pytest.raises(TypeError):
        ops.gather(x, ids, 1.0)


def _off(t, elements):
    """The same shape `elements` behind a 64-byte boundary."""
    buf = torch.zeros(t.numel() + elements + 64, dtype=t.dtype)
    skip = -(buf.data_ptr() // t.element_size()) % (64 // t.element_size()) + elements
    return buf[skip:skip + t.numel()].view(t.shape)


def test_operands_off_a_16_byte_boundary_keep_the_direct_loads(kernels):
    """Whole tiles of operands on multiples of four bytes keep the kernels that they get without a look at the addresses, and
    what is asked of those kernels; ragged sizes keep the loads that take any address."""
    a, h, f8 = torch.zeros(256, 256), torch.zeros(512, 512, dtype=torch.bfloat16), torch.zeros(256, 256).to(torch.float8_e4m3fn)
    for off in (0, 1, 3):
        ops.matmul(_off(a, off), a)
        ops.matmul(a, _off(a, off), BM=64, BN=64, BK=32, WM=2, WN=2, WK=2, NBUF=3)
        ops.matmul(_off(h, 2 * off), h, BM=256, BN=256)
        ops.matmul_fp8(_off(f8, 4 * off), f8, 1.0, 1.0, BM=256, BN=256, WM=4)
    assert len(kernels) == 11          # (the first, bound by its key, is asked for once per alignment)
    for family, params in kernels:
        text, _ = R.emit_kernel(family, "kernel0", **params)
        assert "global_load_lds" in text and ("#define GL_" in text or "#define G8_" in text or "#define GB_D2L 1\n" in text), (family, params)
    del kernels[:]
    ops.matmul(_off(h, 1), h)
    ops.matmul(_off(h[:300], 2), h)
    for family, params in kernels:
        text, _ = R.emit_kernel(family, "kernel0", **params)
        assert "#define GB_D2L 1\n" not in text and "#define GB_SHIFT 1\n" not in text, params


def test_options_that_change_the_kernel_are_kept_apart(kernels):
    """Calls on the same shapes that differ in one option each, twice over: every option asks for a kernel of its own, once."""
    x, g = torch.zeros(4, 8), torch.zeros(8)
    q = torch.zeros(1, 2, 64, 64, dtype=torch.float16)
    calls = [lambda: ops.layernorm(x, g, g, 1), lambda: ops.layernorm(x, g, g, 1, eps=1e-6), lambda: ops.layernorm(x, g, g, 1, gelu=True),
             lambda: ops.layernorm(x, g, g[:4], 1), lambda: ops.fmha(q, q, q), lambda: ops.fmha(q, q, q, causal=True),
             lambda: ops.fmha(q, q, q, scale=0.5), lambda: ops.fmha(q, q, q, scale=0.25), lambda: ops.fmha(q, q, q, out_dtype=torch.float32),
             lambda: ops.softmax(x), lambda: ops.softmax(x.clone(), inplace=True), lambda: ops.elementwise(x, "Gelu"),
             lambda: ops.elementwise(x, "Relu"), lambda: ops.elementwise(x, "Relu", inplace=True), lambda: ops.binary(x, x, "Add"),
             lambda: ops.binary(x, x, "Sub"), lambda: ops.binary(x, g, "Add"), lambda: ops.matmul(x, x.t().contiguous()),
             lambda: ops.matmul(x, x, trans_b=True), lambda: ops.matmul(x.t().contiguous(), x.t().contiguous(), trans_a=True)]
    for call in calls + calls:
        call()
    assert len(kernels) == len(calls)
    assert len({(f, tuple(sorted(p.items()))) for f, p in kernels}) == len(calls)
