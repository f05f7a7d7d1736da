"""Operator-level convenience wrappers: emit the gfx950 kernel for one
operator instance, compile it once, launch it on torch device tensors.
Shapes are static (baked into the kernel), like every kernel the generator
emits."""
import math
import operator

import torch

from . import runtime as R


def _need_cuda(*ts):
    for t in ts:
        if not (t.is_cuda and t.is_contiguous()):
            raise ValueError("operands must be contiguous device tensors")


# (operator, every property of the operands that the kernel depends on) -> the bound launch of that kernel.  Nothing in a
# key or a value belongs to one tensor: shapes, types, options and whether the operands are aligned.  A call with kernel
# parameters of its own (cfg) goes through get_kernel each time.
_bound = {}


def _into(run, shape=None, dtype=None):
    """A bound launch whose last pointer is the result: a function of the operand tensors (and numbers) that allocates the result,
    of that shape and type on the first operand's device, or like the first operand, launches and returns it.  The result is a plain
    tensor; where a subclass of the operand decides about it (torch.empty_like), the caller allocates."""
    native = getattr(run, "result", None)
    if native is not None:
        return native(shape, dtype)

    def call(*operands):
        first = operands[0]
        out = torch.empty_like(first) if shape is None else torch.empty(shape, dtype=dtype, device=first.device)
        pointers = [t.data_ptr() for t in operands if isinstance(t, torch.Tensor)]
        run(*pointers, out.data_ptr(), *operands[len(pointers):])
        return out
    return call


# storage type of the row kernels (their arithmetic is fp32 throughout): the kernels' F16 parameter
_STORAGE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}


def layernorm(x, gamma, beta, axis, eps=1e-5, gelu=False, out=None, **cfg):
    _need_cuda(x, gamma, beta)
    # plain numbers: a key must not hold an object that can change, nor find 1 for a refused 1.0
    axis, eps, gelu = operator.index(axis), float(eps), int(gelu)
    key = ("layernorm", x.shape, x.dtype, gamma.shape, gamma.dtype, beta.shape, beta.dtype, axis, eps, gelu)
    hit = None if cfg else _bound.get(key)
    if hit is None:
        run = _layernorm_kernel(x, gamma, beta, axis, eps, gelu, cfg).bind()
        hit = run, _into(run)
        if not cfg:
            _bound[key] = hit
    if out is None:
        if type(x) is torch.Tensor:
            return hit[1](x, gamma, beta)
        out = torch.empty_like(x)
    hit[0](x.data_ptr(), gamma.data_ptr(), beta.data_ptr(), out.data_ptr())
    return out


def _layernorm_kernel(x, gamma, beta, axis, eps, gelu, cfg):
    axis = axis + x.dim() if axis < 0 else axis
    rows = int(math.prod(x.shape[:axis])) if axis > 0 else 1
    n = x.numel() // rows
    if x.dtype not in _STORAGE or gamma.dtype != x.dtype or beta.dtype != x.dtype:
        raise ValueError("the LayerNorm kernel takes fp32, IEEE half or bfloat16 tensors of one type")
    return R.get_kernel("layernorm", ROWS=rows, N=n, NG=gamma.numel(), NB=beta.numel(), EPS=float(eps),
                        GELU=int(gelu), F16=_STORAGE[x.dtype], **cfg)


_CTYPE = {torch.float32: "float", torch.int32: "int", torch.float16: "_Float16", torch.bfloat16: "__bf16"}


def elementwise(x, op, inplace=False, out_dtype=None, **cfg):
    _need_cuda(x)
    out_dtype, inplace = out_dtype or x.dtype, int(inplace)
    key = ("elementwise", x.numel(), op, inplace, x.dtype, out_dtype)
    hit = None if cfg else _bound.get(key)
    if hit is None:
        run = R.get_kernel("elementwise", N=x.numel(), OP=op, INPLACE=int(inplace), IN_T=_CTYPE[x.dtype],
                           OUT_T=_CTYPE[out_dtype], **cfg).bind()
        hit = run, None if inplace or out_dtype != x.dtype else _into(run)
        if not cfg:
            _bound[key] = hit
    run, into = hit
    if inplace:
        run(x.data_ptr())
        return x if out_dtype == x.dtype else x.view(out_dtype)
    if into is not None and type(x) is torch.Tensor:
        return into(x)
    y = torch.empty(x.shape, dtype=out_dtype, device=x.device)
    run(x.data_ptr(), y.data_ptr())
    return y


def _aligned(a, b):
    """What both operands' addresses are multiples of: 16, 4, or less (1)."""
    low = a.data_ptr() | b.data_ptr()
    return 1 if low & 3 else 4 if low & 15 else 16


def _alignment(aligned):
    """The kernel parameters for it.  Direct loads into LDS take any address that is a multiple of four bytes, so those give
    the kernels that whole tiles get without looking (fp32 1024^3 off a 16-byte boundary: 21 us, 26 through registers; bf16
    4096^3 with row-major weights: 112 and 129); the forms for all sizes split rows into 16-byte chunks and are for ALIGN = 16.
    Other addresses go through registers."""
    return {"ALIGN": 16} if aligned == 16 else {} if aligned == 4 else {"D2L": 0}


_FAMILY = {torch.float32: "gemm_f32", torch.float64: "gemm_f64", torch.bfloat16: "gemm_bf16", torch.float16: "gemm_bf16"}


def batched_matmul(a, b, trans_a=False, trans_b=False, out_dtype=None, **cfg):
    """a: [..., m, k] (or [..., k, m] when trans_a), b: [..., k, n] (or [..., n, k]).  out_dtype None: fp64 for fp64
    operands, fp32 for all others; a type the operands' kernel family does not write raises."""
    _need_cuda(a, b)
    trans_a, trans_b = bool(trans_a), bool(trans_b)
    key = ("matmul", a.shape, b.shape, a.dtype, b.dtype, trans_a, trans_b, out_dtype, _aligned(a, b))
    hit = None if cfg else _bound.get(key)
    if hit is None:
        hit = _matmul_launch(a, b, trans_a, trans_b, out_dtype, cfg)
        if not cfg:
            _bound[key] = hit
    return hit(a, b)


def _matmul_launch(a, b, trans_a, trans_b, out_dtype, cfg):
    """The bound kernel, which allocates its result."""
    if a.dtype != b.dtype or a.dtype not in _FAMILY:
        raise ValueError("unsupported operand dtypes")
    batch = int(math.prod(a.shape[:-2])) if a.dim() > 2 else 1
    m, k = (a.shape[-1], a.shape[-2]) if trans_a else (a.shape[-2], a.shape[-1])
    n, k2 = (b.shape[-2], b.shape[-1]) if trans_b else (b.shape[-1], b.shape[-2])
    if k != k2:
        raise ValueError("incompatible K dimensions")
    extra, align = {}, {}
    if out_dtype is None:
        out_dtype = torch.float64 if a.dtype == torch.float64 else torch.float32
    if a.dtype in (torch.bfloat16, torch.float16):
        if out_dtype not in (torch.float32, a.dtype):
            raise ValueError("a 16-bit GEMM writes fp32 or its operands' type")
        extra["OUT_BF16"] = int(out_dtype == a.dtype)       # a 16-bit result, of the operands' type
        if a.dtype == torch.float16:
            extra["F16"] = 1
        align = _alignment(_aligned(a, b))
    elif a.dtype == torch.float64:
        if out_dtype != torch.float64:
            raise ValueError("fp64 GEMM writes fp64")
    elif out_dtype != torch.float32:
        raise ValueError("fp32 GEMM writes fp32")
    else:
        align = _alignment(_aligned(a, b))
    # (the caller's parameters go before the alignment's, and may not name any other)
    kern = R.get_kernel(_FAMILY[a.dtype], M=m, N=n, K=k, BATCH=batch, TA=int(trans_a), TB=int(trans_b),
                        **extra, **{**align, **cfg})
    run = (lambda *p: kern.launch(*p)) if kern.info["workspace_bytes"] else kern.bind()
    return _into(run, tuple(a.shape[:-2]) + (m, n), out_dtype)


def matmul_fp8(a, b, scale_a, scale_b, trans_a=False, trans_b=True, out_dtype=torch.float32, **cfg):
    """(scale_a * op(a)) (scale_b * op(b)) with fp8 e4m3 operands, one fp32 scale per tensor and fp32
    accumulation.  a: [..., m, k] (or [..., k, m] when trans_a), b: [..., k, n] (or [..., n, k] when
    trans_b, the default: both operands k-contiguous, no transposition on the way into LDS)."""
    _need_cuda(a, b)
    trans_a, trans_b = bool(trans_a), bool(trans_b)
    key = ("matmul_fp8", a.shape, b.shape, a.dtype, b.dtype, trans_a, trans_b, out_dtype, _aligned(a, b))
    hit = None if cfg else _bound.get(key)
    if hit is None:
        hit = _matmul_fp8_launch(a, b, trans_a, trans_b, out_dtype, cfg)
        if not cfg:
            _bound[key] = hit
    return hit(a, b, float(scale_a), float(scale_b))


def _matmul_fp8_launch(a, b, trans_a, trans_b, out_dtype, cfg):
    if a.dtype != torch.float8_e4m3fn or b.dtype != torch.float8_e4m3fn:
        raise ValueError("operands must be float8_e4m3fn")
    if out_dtype not in (torch.float32, torch.bfloat16):
        raise ValueError("output must be fp32 or bf16")
    batch = int(math.prod(a.shape[:-2])) if a.dim() > 2 else 1
    m, k = (a.shape[-1], a.shape[-2]) if trans_a else (a.shape[-2], a.shape[-1])
    n, k2 = (b.shape[-2], b.shape[-1]) if trans_b else (b.shape[-1], b.shape[-2])
    if k != k2:
        raise ValueError("incompatible K dimensions")
    kern = R.get_kernel("gemm_fp8", M=m, N=n, K=k, BATCH=batch, TA=int(trans_a), TB=int(trans_b),
                        OUT_BF16=int(out_dtype == torch.bfloat16), **{**_alignment(_aligned(a, b)), **cfg})
    return _into(kern.bind(scalars=2), tuple(a.shape[:-2]) + (m, n), out_dtype)


def matmul(a, b, **cfg):
    return batched_matmul(a, b, **cfg)


def fmha(q, k, v, scale=None, causal=False, out_dtype=None, **cfg):
    """softmax(scale * q k^T [+ causal mask]) v over [B, H, S, D] operands, all fp32, all bf16 or all IEEE half; the
    result has their type (default) or is fp32.  fp32 operands run both products on the fp32 MFMA (fmha_f32)."""
    _need_cuda(q, k, v)
    if q.dim() != 4 or q.shape != k.shape or q.shape != v.shape:
        raise ValueError("q, k, v must share one [B, H, S, D] shape")
    if not (q.dtype == k.dtype == v.dtype and q.dtype in (torch.float32, torch.bfloat16, torch.float16)):
        raise ValueError("the fused attention kernels take fp32, bf16 or IEEE half operands")
    out_dtype = q.dtype if out_dtype is None else out_dtype
    if out_dtype not in (q.dtype, torch.float32):
        raise ValueError("output must have the operands' type or be fp32")
    scale, causal = (None if scale is None else float(scale)), int(causal)
    key = ("fmha", q.shape, q.dtype, scale, causal, out_dtype)
    run = None if cfg else _bound.get(key)
    if run is None:
        b, h, s, d = q.shape
        scale = d ** -0.5 if scale is None else scale
        if q.dtype == torch.float32:
            kern = R.get_kernel("fmha_f32", B=b, H=h, S=s, D=d, CAUSAL=int(causal), SCALE=scale, **{"FILL": 1, **cfg})
        else:
            kern = R.get_kernel("fmha_bf16", B=b, H=h, S=s, D=d, CAUSAL=int(causal), SCALE=scale,
                                OUT_BF16=int(out_dtype == q.dtype), F16=int(q.dtype == torch.float16), **{"FILL": 1, **cfg})
        run = _into(kern.bind(), tuple(q.shape), out_dtype)
        if not cfg:
            _bound[key] = run
    return run(q, k, v)


def binary(x, y, op, inplace=False, **cfg):
    """x op y (Add, Sub, Mul, Div, Pow; Equal and Greater give a bool tensor) on two fp32 or two IEEE half tensors
    with numpy-style broadcasting."""
    _need_cuda(x, y)
    if x.dtype not in (torch.float32, torch.float16) or y.dtype != x.dtype:
        raise ValueError("the binary kernel takes two fp32 or two IEEE half operands")
    inplace = int(inplace)
    key = ("binary", x.shape, y.shape, x.dtype, op, inplace)
    hit = None if cfg else _bound.get(key)
    if hit is None:
        hit = _binary_launch(x, y, op, inplace, cfg)
        if not cfg:
            _bound[key] = hit
    if inplace:
        hit(x.data_ptr(), y.data_ptr())
        return x
    return hit(x, y)


def _binary_launch(x, y, op, inplace, cfg):
    shape = torch.broadcast_shapes(x.shape, y.shape)

    def strides(t):
        out, run = [0] * len(shape), 1
        for i in range(t.dim()):
            extent = t.shape[t.dim() - 1 - i]
            if extent != 1:
                out[len(shape) - 1 - i] = run
            run *= extent
        return ",".join(map(str, out))

    k = R.get_kernel("binary", OP=op, DIMS=",".join(map(str, shape)), SA=strides(x), SB=strides(y), INPLACE=int(inplace),
                     F16=int(x.dtype == torch.float16), **cfg)
    return k.bind() if inplace else _into(k.bind(), tuple(shape), torch.bool if op in ("Equal", "Greater") else x.dtype)


def gather(x, indices, axis=0, **cfg):
    """out[o.., i.., r..] = x[o.., indices[i..], r..]: dimension `axis` of x is replaced by the dimensions of
    `indices` (int64; a single index, shape (1,), drops the dimension).  Indices outside the axis are clamped.
    `cfg` overrides kernel parameters (BLOCK, UNROLL)."""
    _need_cuda(x, indices)
    if indices.dtype != torch.int64:
        raise ValueError("gather indices must be int64")
    axis = operator.index(axis)
    if not -x.dim() <= axis < x.dim():
        raise ValueError("axis out of range")
    key = ("gather", x.shape, x.dtype, indices.shape, axis)
    hit = None if cfg else _bound.get(key)
    if hit is None:
        hit = _gather_launch(x, indices, axis, cfg)
        if not cfg:
            _bound[key] = hit
    return hit(x, indices)


def _gather_launch(x, indices, axis, cfg):
    axis %= x.dim()
    outer = 1
    for d in x.shape[:axis]:
        outer *= d
    inner = 1
    for d in x.shape[axis + 1:]:
        inner *= d
    single = tuple(indices.shape) == (1,)
    shape = tuple(x.shape[:axis]) + (() if single else tuple(indices.shape)) + tuple(x.shape[axis + 1:])
    kern = R.get_kernel("gather", OUTER=outer, AXIS=x.shape[axis], NIDX=indices.numel(), INNER=inner, ESIZE=x.element_size(), **cfg)
    return _into(kern.bind(), shape, x.dtype)


def softmax(x, inplace=False):
    """softmax over the last axis of an fp32, IEEE half or bfloat16 tensor (fp32 arithmetic)."""
    _need_cuda(x)
    if x.dtype not in _STORAGE:
        raise ValueError("the softmax kernel takes fp32, IEEE half or bfloat16 operands")
    inplace = int(inplace)
    key = ("softmax", x.shape, x.dtype, inplace)
    hit = _bound.get(key)
    if hit is None:
        n = x.shape[-1]
        run = R.get_kernel("softmax", ROWS=x.numel() // n, N=n, INPLACE=int(inplace), F16=_STORAGE[x.dtype]).bind()
        _bound[key] = hit = run, None if inplace else _into(run)
    if inplace:
        hit[0](x.data_ptr())
        return x
    if type(x) is torch.Tensor:
        return hit[1](x)
    y = torch.empty_like(x)
    hit[0](x.data_ptr(), y.data_ptr())
    return y

