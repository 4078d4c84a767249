"""Causal rotary attention (lm_ops.rotary_attention) against the same in fp64 on the same bf16 inputs, forward and
gradient. The probabilities, score gradients, rotated q and k and the results are rounded to bf16 (2^-9 of a value on
average over its rounding), the sums are fp32: norm-relative 1e-2, the bar of every bf16 path here, and no further from
fp64 than torch's flash attention by more than a tenth (its own roundings are the same, the order of sums not). Sizes:
one token, around a wave's 32 rows, a tile's 64, a workgroup's 128, several of each; one head, an odd count, more than
the eight XCDs' turn."""
import pytest
import torch

from gpu_helpers import DEV

pytestmark = pytest.mark.gpu


def reference(qkv, heads, theta=1e6):
    b, t, _ = qkv.shape
    q, k, v = qkv.view(b, t, 3, heads, 64).permute(2, 0, 3, 1, 4).unbind(0)
    f = torch.outer(torch.arange(t, device=qkv.device, dtype=torch.float32),
                    1.0 / theta ** (torch.arange(0, 64, 2, device=qkv.device, dtype=torch.float32) / 64))
    cos, sin = (torch.cat((x, x), -1).bfloat16().to(qkv.dtype) for x in (f.cos(), f.sin()))
    rot = lambda x: x * cos + torch.cat((-x[..., 32:], x[..., :32]), -1) * sin
    s = (rot(q) @ rot(k).transpose(-1, -2).contiguous()) / 8
    s = s.masked_fill(torch.ones(t, t, dtype=torch.bool, device=qkv.device).triu(1), float("-inf"))
    return (torch.softmax(s, -1) @ v.contiguous()).transpose(1, 2).reshape(b, t, heads * 64)


def rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


@pytest.mark.parametrize("b,t,heads", [(1, 1, 1), (2, 2, 3), (1, 31, 2), (1, 33, 1), (2, 64, 4), (1, 65, 9), (3, 127, 3),
                                       (1, 128, 12), (2, 129, 5), (1, 321, 8), (2, 1025, 3)])
@pytest.mark.parametrize("spread", [1.0, 6.0])
def test_rotary_attention(b, t, heads, spread):
    from loopback_amd import lm, lm_ops as ops
    print(f"case attention b{b} t{t} heads{heads} spread{spread}", flush=True)
    g = torch.Generator().manual_seed(t + heads)
    x = (torch.randn(b, t, 3 * heads * 64, generator=g) * spread).bfloat16().to(DEV).requires_grad_()
    dy = torch.randn(b, t, heads * 64, generator=g).bfloat16().to(DEV)
    att = lm.Attention(lm.LMConfig(hidden_size=64 * heads, num_heads=heads)).to(DEV)
    assert ops.attention_native(x, 64)
    cos, sin = att.rotary.tables(t, x.device, x.dtype)
    y = ops.rotary_attention(x, cos, sin, heads, att.attend)
    y.backward(dy)
    torch.cuda.synchronize()
    x64 = x.detach().double().requires_grad_()
    y64 = reference(x64, heads)
    y64.backward(dy.double())
    xt = x.detach().clone().requires_grad_()
    yt = att.attend(xt)
    yt.backward(dy)
    assert rel(y, y64) <= max(1e-2, 1.1 * rel(yt, y64)), (rel(y, y64), rel(yt, y64))
    if t > 1:   # (one token: q and k take no gradient)
        e, et = rel(x.grad, x64.grad), rel(xt.grad, x64.grad)
        assert e <= max(1e-2, 1.1 * et), (e, et)
    # each of q, k, v on its own (with nearly one-hot rows q's and k's gradients are differences of almost equal values,
    # which both attentions take from the rounded output: then no further than 1.5 times torch's)
    thirds = lambda z: z.view(b, t, 3, -1).unbind(2)[0 if t > 1 else 2:]
    for a, r, u in zip(thirds(x.grad), thirds(x64.grad), thirds(xt.grad)):
        assert rel(a, r) <= max(2e-2, 1.5 * rel(u, r)), (rel(a, r), rel(u, r))


def test_attention_module_paths():
    """The module takes the kernels for bf16 at head width 64 and torch's attention elsewhere, with close results, and
    is deterministic; a hooked rotary module is called."""
    from loopback_amd import lm
    torch.manual_seed(0)
    att = lm.Attention(lm.LMConfig(hidden_size=256, num_heads=4)).to(DEV, torch.bfloat16)
    x = torch.randn(2, 200, 256, device=DEV).bfloat16()
    y = att(x)
    assert torch.equal(y, att(x))
    seen = []
    att.rotary.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    assert rel(att(x), y.double()) <= 1e-2 and len(seen) == 1
    wide = lm.Attention(lm.LMConfig(hidden_size=256, num_heads=2)).to(DEV, torch.bfloat16)
    assert wide(x).shape == x.shape
