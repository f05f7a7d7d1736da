"""Bound launches follow torch's current stream: on a stream of the caller's, in a second thread, and under capture."""
import threading

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from kernelcodegen_amd import ops as _ops
    from kernelcodegen_amd._lib import lib, check
    check(lib().kcg_hip_init(0), "kcg_hip_init")
    return _ops


def _chain(ops, x, g, w):
    """Four operators, each on the result of the one before."""
    y = ops.layernorm(x, g, g, -1)
    y = ops.matmul(y, w, trans_b=True, out_dtype=torch.float16)
    y = ops.elementwise(y, "Gelu")
    return ops.softmax(y)


def _case(seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((64, 512), generator=gen, device="cuda").half()
    return x, torch.ones(512, device="cuda").half(), torch.randn((256, 512), generator=gen, device="cuda").half() * 0.05


def test_launches_on_the_callers_stream_see_its_work(ops):
    """The input is written on the stream behind a product that takes milliseconds: launches on another stream would read what
    was there before."""
    src, g, w = _case(1)
    want = _chain(ops, src, g, w)          # binds the launches, on the default stream
    x, a = torch.zeros_like(src), torch.randn((4096, 4096), device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(4):
            a = a @ a * 1e-4
        x.copy_(src)
        got = _chain(ops, x, g, w)
    stream.synchronize()
    assert torch.equal(got, want)


def test_two_threads_with_streams_of_their_own(ops):
    cases = [_case(seed) for seed in (2, 3)]
    want = [_chain(ops, *c) for c in cases]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(50):
                    got = _chain(ops, *cases[i])
                    torch.cuda.current_stream().synchronize()
                    if not torch.equal(got, want[i]):
                        bad.append(i)
        except Exception as e:      # a thread's own exceptions reach nobody
            bad.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad


def test_bound_launches_are_captured_and_replayed(ops):
    x, g, w = _case(4)
    want = [_chain(ops, x, g, w)]
    other = _case(5)[0]
    want.append(_chain(ops, other, g, w))
    static = x.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _chain(ops, static, g, w)
    for i in (0, 1, 0, 1):
        static.copy_((x, other)[i])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[i]), i
        assert torch.equal(_chain(ops, (x, other)[i], g, w), want[i])


def test_options_of_one_shape_give_their_own_results(ops):
    """eps, scale, mask and the fused GELU separate the bound launches of one shape: each call against fp64."""
    x, g, _ = _case(6)
    x64 = x.double()
    c = x64 - x64.mean(-1, keepdim=True)
    gen = torch.Generator(device="cuda").manual_seed(7)
    q, k, v = (torch.randn((1, 2, 128, 64), generator=gen, device="cuda").half() for _ in range(3))
    for _ in range(2):
        for eps in (1e-5, 1.0):
            want = c / torch.sqrt((c * c).mean(-1, keepdim=True) + eps)
            assert ((ops.layernorm(x, g, g * 0, -1, eps=eps).double() - want).norm() <= 2 ** -10 * want.norm()).item()
            gelu = 0.5 * want * (1 + torch.tanh(0.797884 * (want + 0.044715 * want ** 3)))
            assert ((ops.layernorm(x, g, g * 0, -1, eps=eps, gelu=True).double() - gelu).norm() <= 2 ** -10 * gelu.norm()).item()
        for scale in (0.125, 0.5):
            for causal in (False, True):
                s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * scale
                if causal:
                    s.masked_fill_(torch.ones((128, 128), dtype=torch.bool, device="cuda").triu(1), float("-inf"))
                want = torch.softmax(s, -1) @ v.double()
                # the tolerance of the other 16-bit attention tests: probabilities rounded to 11 bits, fp32 sums
                assert ((ops.fmha(q, k, v, scale=scale, causal=causal).double() - want).norm() <= 2e-3 * want.norm()).item()
