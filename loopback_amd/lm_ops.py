"""The language model's row operations on the HIP kernels of libloopback_lm.so (include/loopback_lm.h): RMSNorm with the
residual's add before it and the residual's gradient folded into its backward, SwiGLU, the next-token cross entropy on
16-bit logits, causal rotary attention in bf16 at head width 64, and the weight gradients of the linear layers.

`native(...)` says whether the kernels take a call: plain 16-bit tensors of one dtype on the current GPU (a launch on
another GPU's default stream would run on the current one), no transform or tracer that has to see torch operations
(torch.func, forward-mode AD, torch.compile, jit tracing, a dispatch mode such as make_fx's), no autocast. Everything
else -- the CPU, fp32, other shapes -- stays on torch in lm.py. A backward that is itself differentiated (create_graph),
that one of these watches or that gets batched gradients runs the torch form of the operation.
"""
from __future__ import annotations

import ctypes
import os

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from . import build as _build

ABI_VERSION = 1
NORM_MAX_WIDTH = 2048
_CODES = {torch.bfloat16: 1, torch.float16: 2}

_p, _i64, _i32, _f32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_float
# name -> (restype, argtypes); one line per declaration of include/loopback_lm.h
SIGNATURES = {
    "llm_abi_version": (_i32, []),
    "llm_rms_norm_fwd": (_i32, [_p, _p, _p, _p, _p, _p, _i64, _i64, _f32, _i32, _p]),
    "llm_rms_norm_parts": (_i64, [_i64]),
    "llm_rms_norm_bwd": (_i32, [_p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i32, _p]),
    "llm_sum_rows": (_i32, [_p, _i64, _i64, _p, _i32, _p]),
    "llm_swiglu_fwd": (_i32, [_p, _p, _i64, _i64, _i32, _p]),
    "llm_swiglu_bwd": (_i32, [_p, _p, _p, _i64, _i64, _i32, _p]),
    "llm_next_token_loss_fwd": (_i32, [_p, _p, _p, _p, _p, _i64, _i64, _i64, _i32, _p]),
    "llm_next_token_loss_bwd": (_i32, [_p, _p, _p, _p, _p, _i64, _i64, _i64, _i32, _p]),
    "llm_rotary": (_i32, [_p, _p, _p, _p, _i64, _i64, _i64, _p]),
    "llm_attn_fwd": (_i32, [_p, _p, _p, _p, _i64, _i64, _i64, _p]),
    "llm_wgrad_splits": (_i64, [_i64, _i64, _i64]),
    "llm_wgrad": (_i32, [_p, _p, _p, _p, _i64, _i64, _i64, _p]),
    "llm_attn_bwd": (_i32, [_p, _p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _p]),
}


def _load() -> ctypes.CDLL:
    path = _build.LM_LIB
    if not os.path.exists(path):
        raise ImportError(f"loopback_lm: {path} is not built (run `python -m loopback_amd.build`)")
    lib = ctypes.CDLL(path)
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)          # AttributeError -> the library is stale
        fn.restype, fn.argtypes = res, args
    if lib.llm_abi_version() != ABI_VERSION:
        raise ImportError(f"loopback_lm: {path} has ABI {lib.llm_abi_version()}, expected {ABI_VERSION}; rebuild")
    return lib


LIB = _load()
_FN = {name: getattr(LIB, name) for name in SIGNATURES}
_raw_stream = torch._C._cuda_getCurrentRawStream


def _run(name: str, *args) -> None:
    code = _FN[name](*args)
    if code:
        raise RuntimeError(f"{name}: refused or failed to launch (code {code})")


def _stream(t: torch.Tensor) -> int:
    return _raw_stream(t.device.index)


_Tensor, _Parameter = torch.Tensor, torch.nn.Parameter   # bound once: these run a few times per layer and pass
_compiling, _tracing, _grad_on = torch.compiler.is_compiling, torch._C._is_tracing, torch.is_grad_enabled
_modes, _transform = torch._C._len_torch_dispatch_stack, torch._C._functorch.peek_interpreter_stack
_batched = torch._C._functorch.is_legacy_batchedtensor


def _watched() -> bool:
    """Whether something is on that has to see torch operations: torch.compile, jit tracing, a torch.func transform,
    forward-mode AD, a dispatch mode."""
    return (_compiling() or _tracing() or forward_ad._current_level >= 0 or _modes() > 0
            or _transform() is not None)


def native(*tensors) -> bool:
    # what watches the call first, then what the arguments are: a tracer's arguments (fake tensors, proxies) are not
    # asked for a device, and a compiler meets no query of the GPU
    if _watched():
        return False
    first = tensors[0]
    for t in tensors:
        if type(t) is not _Tensor and type(t) is not _Parameter:
            return False
    if not first.is_cuda or first.dtype not in _CODES or first.device.index != torch._C._cuda_getDevice():
        return False
    for t in tensors[1:]:
        if t.dtype is not first.dtype or t.device != first.device:
            return False
    return not torch.is_autocast_enabled("cuda")


def _launchable(*grads) -> bool:
    """Whether a backward runs on the kernels: it is not itself differentiated, nothing watches it, and its gradients
    are plain tensors (not the batched ones of is_grads_batched and jacobian(vectorize=True))."""
    if _grad_on() or _watched():
        return False
    for g in grads:
        if g is not None and ((type(g) is not _Tensor and type(g) is not _Parameter) or _batched(g)):
            return False
    return True


def _saved(ctx):
    """The saved tensors as the kernels take them: a saved-tensor hook may give one back with other strides or another
    alignment than it was saved with."""
    ts = ctx.saved_tensors
    return ts if _rows_ok(*ts) else [t if _rows_ok(t) else t.clone(memory_format=torch.contiguous_format) for t in ts]


def _again(fn, inputs, needed, grad):
    """The gradients of fn at `inputs` as torch forms them, with a graph where this backward is differentiated."""
    wanted = [x for x, need in zip(inputs, needed) if need]
    if not wanted:
        return [None] * len(needed)
    graph = torch.is_grad_enabled()
    with torch.enable_grad():
        got = iter(torch.autograd.grad(fn(*inputs), wanted, grad, create_graph=graph))
    return [next(got) if need else None for need in needed]


# ---------------------------------------------------------------------------------------------------------------
# RMSNorm
# ---------------------------------------------------------------------------------------------------------------
class _AddRmsNorm(torch.autograd.Function):
    """(h, y) = (x + add, rms_norm(x + add) w); add may be None (h is then x itself, as an alias). h carries the
    residual stream on, so the gradient that comes back along it joins the norm's in one kernel."""

    @staticmethod
    def forward(ctx, x, add, w, eps):
        d = x.shape[-1]
        rows = x.numel() // d
        h = x.view_as(x) if add is None else torch.empty_like(x)
        y = torch.empty_like(x)
        rstd = torch.empty(rows, device=x.device, dtype=torch.float32)
        _run("llm_rms_norm_fwd", x.data_ptr(), None if add is None else add.data_ptr(), w.data_ptr(),
             None if add is None else h.data_ptr(), y.data_ptr(), rstd.data_ptr(), rows, d, eps, _CODES[x.dtype],
             _stream(x))
        ctx.eps, ctx.added = eps, add is not None
        ctx.save_for_backward(x if add is None else h, w, rstd)
        ctx.set_materialize_grads(False)
        if not (ctx.needs_input_grad[0] or ctx.needs_input_grad[1]):
            ctx.mark_non_differentiable(h)   # only the weight is trained: the residual stream needs no gradient
        return h, y

    @staticmethod
    def backward(ctx, dh, dy):
        h, w, rstd = _saved(ctx)
        if dy is None:
            return dh, dh if ctx.added else None, None, None
        need = ctx.needs_input_grad
        needed = need[0] or need[1], need[2]
        if not _launchable(dh, dy):
            dx, dw = _again(lambda h, w: F.rms_norm(h, (h.shape[-1],), w, ctx.eps), [h, w], needed, dy)
            dx = dx if dx is None or dh is None else dx + dh
            return dx, dx if ctx.added else None, dw, None
        d = h.shape[-1]
        rows = h.numel() // d
        dy = _dense(dy, h)
        dres = None if dh is None else _dense(dh, h)
        dx = torch.empty_like(h) if needed[0] else None
        dw = part = None
        if needed[1]:
            parts = LIB.llm_rms_norm_parts(rows)
            part = torch.empty((parts, d), device=h.device, dtype=torch.float32)
            dw = torch.empty_like(w)
        _run("llm_rms_norm_bwd", dy.data_ptr(), h.data_ptr(), w.data_ptr(), rstd.data_ptr(),
             None if dres is None else dres.data_ptr(), None if dx is None else dx.data_ptr(),
             None if part is None else part.data_ptr(), rows, d, _CODES[h.dtype], _stream(h))
        if needed[1]:
            _run("llm_sum_rows", part.data_ptr(), parts, d, dw.data_ptr(), _CODES[w.dtype], _stream(h))
        return dx, dx if ctx.added else None, dw, None


def _dense(g, like):
    """A gradient as the kernels take it: contiguous rows, 16-byte aligned, the saved tensor's dtype."""
    g = g.to(like.dtype).contiguous()
    return g if g.data_ptr() % 16 == 0 else g.clone()


def _rows_ok(*tensors) -> bool:
    for t in tensors:
        if not t.is_contiguous() or t.data_ptr() % 16:
            return False
    return True


def norm_native(x, w, add=None, eps=0.0) -> bool:
    """Whether add_rms_norm takes the call: rows of a multiple of 8 elements up to NORM_MAX_WIDTH, contiguous; eps given
    (None, the type's epsilon, is torch's to choose)."""
    if eps is None:
        return False
    ts = (x, w) if add is None else (x, w, add)
    if not native(*ts):
        return False
    d = x.shape[-1] if x.dim() else 0
    return (8 <= d <= NORM_MAX_WIDTH and d % 8 == 0 and w.shape == (d,)
            and (add is None or add.shape == x.shape) and _rows_ok(*ts))


def add_rms_norm(x, add, w, eps):
    return _AddRmsNorm.apply(x, add, w, float(eps))


# ---------------------------------------------------------------------------------------------------------------
# SwiGLU
# ---------------------------------------------------------------------------------------------------------------
def _swiglu_torch(gu):
    g, u = gu.chunk(2, dim=-1)
    return F.silu(g) * u


class _SwiGLU(torch.autograd.Function):
    @staticmethod
    def forward(ctx, gu):
        n = gu.shape[-1] // 2
        rows = gu.numel() // (2 * n)
        act = torch.empty((*gu.shape[:-1], n), device=gu.device, dtype=gu.dtype)
        _run("llm_swiglu_fwd", gu.data_ptr(), act.data_ptr(), rows, n, _CODES[gu.dtype], _stream(gu))
        ctx.save_for_backward(gu)
        return act

    @staticmethod
    def backward(ctx, da):
        gu, = _saved(ctx)
        if not _launchable(da):
            return _again(_swiglu_torch, [gu], [True], da)[0]
        n = gu.shape[-1] // 2
        da = _dense(da, gu)
        dgu = torch.empty_like(gu)
        _run("llm_swiglu_bwd", gu.data_ptr(), da.data_ptr(), dgu.data_ptr(), gu.numel() // (2 * n), n,
             _CODES[gu.dtype], _stream(gu))
        return dgu


def swiglu(gu: torch.Tensor) -> torch.Tensor:
    """silu(g) * u of rows [g | u]."""
    if native(gu) and gu.shape[-1] % 16 == 0 and gu.numel() > 0 and _rows_ok(gu):
        return _SwiGLU.apply(gu)
    return _swiglu_torch(gu)


# ---------------------------------------------------------------------------------------------------------------
# next-token cross entropy
# ---------------------------------------------------------------------------------------------------------------
def _loss_torch(ids):
    def fn(logits):
        labels = torch.cat((ids[:, 1:], torch.full_like(ids[:, :1], -100)), dim=1)
        return F.cross_entropy(logits.reshape(-1, logits.shape[-1]).float(), labels.reshape(-1), ignore_index=-100)
    return fn


class _NextTokenLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logits, ids):
        b, t, vocab = logits.shape
        lse = torch.empty((b * t, 2), device=logits.device, dtype=torch.float32)
        scratch = torch.empty(b * t, device=logits.device, dtype=torch.float32)
        loss = torch.empty((), device=logits.device, dtype=torch.float32)
        _run("llm_next_token_loss_fwd", logits.data_ptr(), ids.data_ptr(), lse.data_ptr(), scratch.data_ptr(),
             loss.data_ptr(), b, t, vocab, _CODES[logits.dtype], _stream(logits))
        ctx.save_for_backward(logits, ids, lse)
        return loss

    @staticmethod
    def backward(ctx, g):
        logits, ids, lse = _saved(ctx)
        if not _launchable(g):
            return _again(_loss_torch(ids), [logits], [True], g)[0], None
        b, t, vocab = logits.shape
        dlogits = torch.empty_like(logits)
        _run("llm_next_token_loss_bwd", logits.data_ptr(), ids.data_ptr(), lse.data_ptr(), g.data_ptr(),
             dlogits.data_ptr(), b, t, vocab, _CODES[logits.dtype], _stream(logits))
        return dlogits, None


def next_token_loss(logits: torch.Tensor, ids: torch.Tensor) -> torch.Tensor:
    """Mean cross entropy of logits (b, t, vocab) against ids shifted by one, the last position ignored."""
    if (native(logits) and type(ids) is torch.Tensor and ids.device == logits.device and ids.dtype is torch.int64
            and ids.is_contiguous() and logits.is_contiguous() and logits.shape[:-1] == ids.shape
            and 0 < ids.numel() < 2 ** 31):
        return _NextTokenLoss.apply(logits, ids)
    return _loss_torch(ids)(logits)


# ---------------------------------------------------------------------------------------------------------------
# causal rotary attention
# ---------------------------------------------------------------------------------------------------------------
class _RotaryAttention(torch.autograd.Function):
    """qkv (b, t, 3 heads 64) -> (b, t, heads 64). Saves the rotated q and k, qkv (for v), the output and the queries'
    sums of exponentials. `again`: the torch form, for a backward that is differentiated."""

    @staticmethod
    def forward(ctx, qkv, cos, sin, heads, again):
        b, t, _ = qkv.shape
        qk = torch.empty((b, t, 2, heads, 64), device=qkv.device, dtype=qkv.dtype)
        out = torch.empty((b, t, heads * 64), device=qkv.device, dtype=qkv.dtype)
        lse2 = torch.empty((b * heads, t), device=qkv.device, dtype=torch.float32)
        st = _stream(qkv)
        _run("llm_rotary", qkv.data_ptr(), cos.data_ptr(), sin.data_ptr(), qk.data_ptr(), b, t, heads, st)
        _run("llm_attn_fwd", qk.data_ptr(), qkv.data_ptr(), out.data_ptr(), lse2.data_ptr(), b, t, heads, st)
        ctx.heads, ctx.again = heads, again
        ctx.save_for_backward(qkv, qk, out, lse2, cos, sin)
        return out

    @staticmethod
    def backward(ctx, dout):
        qkv, qk, out, lse2, cos, sin = _saved(ctx)
        if not _launchable(dout):
            return _again(ctx.again, [qkv], [True], dout)[0], None, None, None, None
        b, t, _ = qkv.shape
        dout = _dense(dout, out)
        delta = torch.empty_like(lse2)
        dqkv = torch.empty_like(qkv)
        _run("llm_attn_bwd", qk.data_ptr(), qkv.data_ptr(), out.data_ptr(), dout.data_ptr(), lse2.data_ptr(),
             cos.data_ptr(), sin.data_ptr(), delta.data_ptr(), dqkv.data_ptr(), b, t, ctx.heads, _stream(qkv))
        return dqkv, None, None, None, None


ATTN_MAX = 0x7fffff   # tokens a sequence, and sequences times heads, as llm_attn_fwd checks them


def attention_native(qkv: torch.Tensor, head_dim: int) -> bool:
    """Whether rotary_attention takes qkv (b, t, 3 heads head_dim): bf16, head width 64, not empty, within the
    kernels' index range."""
    return (head_dim == 64 and qkv.dtype is torch.bfloat16 and native(qkv) and qkv.dim() == 3 and qkv.numel() > 0
            and qkv.shape[1] <= ATTN_MAX and qkv.shape[0] * qkv.shape[2] <= 192 * ATTN_MAX and _rows_ok(qkv))


def tables_native(qkv, cos, sin, heads: int) -> bool:
    """Whether the operands have the sizes the kernels index by: qkv's width that of the heads, cos and sin (t, 64)."""
    return qkv.shape[2] == 192 * heads and all(
        type(x) is torch.Tensor and x.dtype is torch.float32 and x.device == qkv.device
        and x.shape == (qkv.shape[1], 64) and _rows_ok(x) for x in (cos, sin))


def rotary_attention(qkv, cos, sin, heads, again):
    """Causal attention over the rotated q and k of qkv; cos and sin (t, 64) fp32, contiguous, both halves alike."""
    return _RotaryAttention.apply(qkv, cos, sin, heads, again)


# ---------------------------------------------------------------------------------------------------------------
# bias-free linear layers, their weight gradient by llm_wgrad
# ---------------------------------------------------------------------------------------------------------------
# Where the split reduction is the faster one, library's time over the kernels': 8192 to 65536 tokens, weights 64 x 64 to
# 4096 x 768 and up to 2056 x 1032: 1.08 to 5.9 (the smallest too, though their tile is mostly padding: the library runs a
# few workgroups). A side of 8 or 16: 0.94 to 1.06 up to 16384 tokens. Four runs of tokens (2048 x 2048, 4096 x 1024): 0.95
# to 1.16; two (5632 x 1024): 0.84. 4096 tokens and fewer: 0.6 to 1.1. The library's then.
WGRAD_MIN_TOKENS, WGRAD_MIN_SPLITS, WGRAD_MIN_SIDE = 8192, 5, 64


def wgrad(dy: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """dy^T x of (tokens, n) and (tokens, k) rows, bf16."""
    (m, n), k = dy.shape, x.shape[1]
    part = torch.empty((LIB.llm_wgrad_splits(m, n, k), n, k), device=x.device, dtype=torch.float32)
    dw = torch.empty((n, k), device=x.device, dtype=x.dtype)
    _run("llm_wgrad", dy.data_ptr(), x.data_ptr(), part.data_ptr(), dw.data_ptr(), m, n, k, _stream(x))
    return dw


class _Linear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        return F.linear(x, w)

    @staticmethod
    def backward(ctx, dy):
        x, w = _saved(ctx)
        if not _launchable(dy):
            return tuple(_again(F.linear, [x, w], ctx.needs_input_grad, dy))
        dy = _dense(dy, x).view(-1, w.shape[0])
        dx = (dy @ w).view(x.shape) if ctx.needs_input_grad[0] else None
        return dx, wgrad(dy, x.view(-1, w.shape[1])) if ctx.needs_input_grad[1] else None


def linear_native(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether linear(x, w) records a weight gradient by llm_wgrad."""
    return (torch.is_grad_enabled() and x.dtype is torch.bfloat16 and not _compiling()
            and w.requires_grad and x.dim() > 1 and w.dim() == 2 and x.shape[-1] == w.shape[1]
            and x.numel() >= WGRAD_MIN_TOKENS * w.shape[1] and min(w.shape) >= WGRAD_MIN_SIDE and w.shape[0] % 8 == 0
            and w.shape[1] % 8 == 0 and native(x, w) and _rows_ok(x, w)
            and LIB.llm_wgrad_splits(x.numel() // w.shape[1], *w.shape) >= WGRAD_MIN_SPLITS)


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """F.linear(x, w), with the weight's gradient by llm_wgrad where that is the faster one."""
    return _Linear.apply(x, w) if linear_native(x, w) else F.linear(x, w)
