"""The native bound launches (launch.cc): what they refuse without a GPU, and what they pass on and return with one."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")

from kernelcodegen_amd import runtime as R

ENTRY = C.CFUNCTYPE(C.c_int, C.c_void_p, C.POINTER(C.c_uint32), C.c_void_p, C.c_void_p, C.c_int)


def _fail(rc):
    raise ValueError("status %d" % rc)


class Entry:
    """Stands for kcg_hip_launch_packed: keeps what it was given and returns `status`."""

    def __init__(self, status=0):
        self.calls, self.status = [], status
        self.function = ENTRY(self._call)
        self.address = C.cast(self.function, C.c_void_p).value

    def _call(self, handle, dims, stream, slots, n):
        self.calls.append((handle, list(dims[:7]), stream, list((C.c_uint64 * n).from_address(slots))))
        return self.status


def make(entry, pointers, scalars):
    kind = R._native_launch()
    assert kind is not None, "the extension is built with the library"
    return kind(entry.address, 77, (1, 2, 3, 64, 1, 1, 9), pointers, scalars, _fail, entry)


def test_wrong_arguments_are_refused():
    entry = Entry()
    run = make(entry, 2, 1)
    for args in ((), (1, 2), (1, 2, 3.0, 4.0), (1, 2, "x"), (-1, 2, 1.0), (1 << 64, 2, 1.0), (1.5, 2, 1.0), (None, 2, 1.0)):
        with pytest.raises((TypeError, OverflowError)):
            run(*args)
    with pytest.raises(TypeError):
        run(1, 2, value=1.0)
    into = run.result((2, 3), torch.float32)
    for args in ((1, 2.0), (torch.zeros(2),), (5, 1.0), (torch.zeros(2), 3, 1.0)):
        with pytest.raises(TypeError):
            into(*args)
    for bad in (((2, 3), None), ((2, 3), 5), (7, torch.float32), (("a",), torch.float32)):
        with pytest.raises(TypeError):
            run.result(*bad)
    kind = R._native_launch()
    for bad in (dict(p=0, s=0), dict(p=17, s=0), dict(p=10, s=7), dict(p=1, s=-1)):
        with pytest.raises(ValueError):
            kind(entry.address, 77, (1, 1, 1, 64, 1, 1, 0), bad["p"], bad["s"], _fail, None)
    assert not entry.calls


def test_a_pointer_is_any_whole_number():
    """What has __index__, as for the ctypes launches."""
    numpy = pytest.importorskip("numpy")
    entry = Entry()
    run = make(entry, 2, 0)
    if torch.cuda.is_available():
        run(numpy.int64(16), numpy.uint64(1 << 63))
        assert entry.calls[-1][3] == [16, 1 << 63]
    else:
        with pytest.raises(RuntimeError):         # (of the stream that is not there, behind the arguments)
            run(numpy.int64(16), numpy.uint64(1 << 63))


def test_without_a_gpu_a_launch_is_an_error():
    if torch.cuda.is_available():
        pytest.skip("there is one")
    entry = Entry()
    with pytest.raises(RuntimeError):
        make(entry, 1, 0)(16)
    with pytest.raises(RuntimeError):
        make(entry, 2, 0).result(None, None)(torch.zeros(4))
    assert not entry.calls


@pytest.mark.parametrize("content", [None, b"no library", "other version"])
def test_an_extension_that_is_missing_or_does_not_fit_gives_way_to_ctypes(tmp_path, monkeypatch, content):
    """No file, one that does not load, and one that loads but was built for another torch."""
    import sys
    import types
    import kernelcodegen_amd
    from kernelcodegen_amd import build as B
    name = "kernelcodegen_amd._launch"
    monkeypatch.setattr(R, "_launch_type", None)
    monkeypatch.setattr(kernelcodegen_amd, "__path__", [str(tmp_path)])
    monkeypatch.delitem(sys.modules, name, raising=False)
    if content == "other version":
        monkeypatch.setitem(sys.modules, name, types.SimpleNamespace(torch_version="1.0", Launch=None))
    elif content is not None:
        (tmp_path / B.os.path.basename(B.LAUNCH)).write_bytes(content)
    if content is None:
        assert R._native_launch() is None
    else:
        with pytest.warns(RuntimeWarning, match="ctypes"):
            assert R._native_launch() is None
    kern = R.Kernel(None, C.c_void_p(5), dict(grid=(1, 1, 1), block=(64, 1, 1), lds_bytes=0, num_args=2, workspace_bytes=0))
    monkeypatch.setattr(R, "_current_stream", lambda: lambda: 0)
    assert not hasattr(kern.bind(), "result") and callable(kern.bind())


def test_the_library_is_built_where_the_extension_cannot_be(tmp_path, monkeypatch, capfd):
    from kernelcodegen_amd import build as B
    compiler, launch = tmp_path / "cxx", tmp_path / "_launch.so"
    compiler.write_text("#!/bin/sh\necho no such header >&2\nexit 1\n")
    compiler.chmod(0o755)
    launch.write_bytes(b"of an earlier build")
    monkeypatch.setattr(B, "LAUNCH", str(launch))
    monkeypatch.setattr(B, "CXX", str(compiler))
    monkeypatch.setattr(B, "build_library", lambda force, verbose: "library")
    assert B.build() == "library" and not launch.exists()
    assert "no such header" in capfd.readouterr().err
    monkeypatch.setitem(__import__("sys").modules, "torch", None)      # no torch at all
    assert B.build() == "library"


@pytest.mark.gpu
def test_what_is_passed_on():
    entry = Entry()
    x = torch.zeros(4, 8, device="cuda")
    side = torch.cuda.Stream()
    run = make(entry, 2, 2)
    with torch.cuda.stream(side):
        assert run(16, x, 0.5, 1e39) is None
    handle, dims, stream, slots = entry.calls[-1]
    assert (handle, dims, stream) == (77, [1, 2, 3, 64, 1, 1, 9], side.cuda_stream)
    bits = [int.from_bytes(bytes(C.c_float(v)), "little") for v in (0.5, 1e39)]
    assert slots == [16, x.data_ptr()] + bits
    y = run.result((3, 5), torch.bfloat16)(x, -1e39, float("nan"))
    assert (y.shape, y.dtype, y.device, y.is_contiguous()) == ((3, 5), torch.bfloat16, x.device, True)
    assert entry.calls[-1][3][:3] == [x.data_ptr(), y.data_ptr(), int.from_bytes(bytes(C.c_float(float("-inf"))), "little")]
    z = make(entry, 3, 0).result(None, None)(torch.nn.Parameter(x), 32)
    assert (z.shape, z.dtype, z.requires_grad, type(z)) == (x.shape, x.dtype, False, torch.Tensor) and entry.calls[-1][3] == [x.data_ptr(), 32, z.data_ptr()]


@pytest.mark.gpu
def test_a_failed_launch_raises():
    x = torch.zeros(4, device="cuda")
    run = make(Entry(5), 2, 0)
    for call in (lambda: run(16, 32), lambda: run.result(None, None)(x)):
        with pytest.raises(ValueError, match="status 5"):
            call()


class Marked(torch.Tensor):
    pass


@pytest.mark.gpu
@pytest.mark.parametrize("wrap,like", [(lambda x: x.as_subclass(Marked), Marked), (lambda x: torch.nn.Parameter(x, requires_grad=False), torch.Tensor)])
def test_a_result_like_the_operand_is_of_its_subclass(wrap, like):
    """What torch.empty_like gives; the other results are plain tensors."""
    from kernelcodegen_amd import ops
    x, one, zero = torch.randn(64, 512, device="cuda"), torch.ones(512, device="cuda"), torch.zeros(512, device="cuda")
    for call, result in [(lambda x: ops.softmax(x), like), (lambda x: ops.layernorm(x, one, zero, 1), like),
                         (lambda x: ops.elementwise(x, "Relu"), torch.Tensor), (lambda x: ops.matmul(x, x.t().contiguous()), torch.Tensor)]:
        got = call(wrap(x))
        assert type(got) is result
        assert torch.equal(got.as_subclass(torch.Tensor), call(x))
