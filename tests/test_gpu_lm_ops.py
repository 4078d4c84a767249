"""The language model's row kernels (lm_ops) against torch in fp64 on the same 16-bit inputs: every result is an fp32
value rounded once, so each element lies within half a unit in the last place (2^-8 of a bf16 value, 2^-11 of an fp16 one)
plus fp32 round-off (1e-5 of the result's RMS). Sizes: one vector, a lane's and a wave's edges, the widest row; one
row, remainders, more rows than workgroups take at once; vocabularies below, at and past a vector and a workgroup's
2048 logits. Then what must stay torch's: second derivatives, hooks on the norms, forward mode, fp32."""
import pytest
import torch
import torch.nn.functional as F

from gpu_helpers import DEV

pytestmark = pytest.mark.gpu
HALF = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}   # significands of 8 and 11 bits: half a step of the last


def close(got, ref, dtype):
    ref = ref.double()
    rms = ref.pow(2).mean().sqrt() if ref.numel() else 0.0
    tiny = 2.0 ** -25 if dtype is torch.float16 else 0.0   # half of fp16's smallest subnormal
    bad = (got.double() - ref).abs() > HALF.get(dtype, 0.0) * ref.abs() + 1e-5 * rms + tiny
    assert not bad.any(), ((got.double() - ref).abs().max().item(), rms)


def rnd(shape, dtype, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


@pytest.mark.parametrize("rows,d", [(1, 8), (5, 16), (3, 512), (7, 520), (2049, 768), (5, 1032), (9, 2048)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("add", [False, True])
def test_add_rms_norm(rows, d, dtype, add):
    from loopback_amd import lm_ops as ops
    print(f"case norm {rows}x{d} {dtype} add={add}", flush=True)
    x, w = rnd((rows, d), dtype, 1).requires_grad_(), rnd((d,), dtype, 2).requires_grad_()
    a = rnd((rows, d), dtype, 3).requires_grad_() if add else None
    dh, dy = rnd((rows, d), dtype, 4), rnd((rows, d), dtype, 5)
    assert ops.norm_native(x, w, a)
    h, y = ops.add_rms_norm(x, a, w, 1e-6)
    torch.autograd.backward((h, y), (dh, dy))
    torch.cuda.synchronize()
    hr = (x + a if add else x).detach()
    assert torch.equal(h, hr)
    h64, w64 = hr.double().requires_grad_(), w.detach().double().requires_grad_()
    y64 = F.rms_norm(h64, (d,), w64, 1e-6)
    torch.autograd.backward((h64, y64), (dh.double(), dy.double()))
    close(y, y64.detach(), dtype)
    close(x.grad, h64.grad, dtype)
    close(w.grad, w64.grad, dtype)
    if add:
        assert torch.equal(a.grad, x.grad)


@pytest.mark.parametrize("rows,n", [(1, 8), (3, 264), (2049, 2048)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_swiglu(rows, n, dtype):
    from loopback_amd import lm_ops as ops
    print(f"case swiglu {rows}x{n} {dtype}", flush=True)
    gu = (3 * rnd((rows, 2 * n), dtype, 6)).requires_grad_()
    da = rnd((rows, n), dtype, 7)
    act = ops.swiglu(gu)
    act.backward(da)
    torch.cuda.synchronize()
    g64 = gu.detach().double().requires_grad_()
    a64 = F.silu(g64[:, :n]) * g64[:, n:]
    a64.backward(da.double())
    close(act, a64.detach(), dtype)
    close(gu.grad, g64.grad, dtype)


@pytest.mark.parametrize("b,t,vocab", [(1, 2, 1), (2, 3, 7), (1, 9, 8), (3, 5, 33), (2, 17, 2048), (2, 4, 2057),
                                       (3, 300, 32000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_next_token_loss(b, t, vocab, dtype):
    from loopback_amd import lm_ops as ops
    print(f"case loss {b}x{t}x{vocab} {dtype}", flush=True)
    ids = torch.randint(0, vocab, (b, t), generator=torch.Generator().manual_seed(8)).to(DEV)
    x = (4 * rnd((b, t, vocab), dtype, 9)).requires_grad_()
    loss = ops.next_token_loss(x, ids)
    (2.0 * loss).backward()
    torch.cuda.synchronize()
    x64 = x.detach().double().requires_grad_()
    l64 = F.cross_entropy(x64[:, :-1].reshape(-1, vocab), ids[:, 1:].reshape(-1))
    (2.0 * l64).backward()
    assert abs(loss.item() - l64.item()) <= 2e-6 * max(1.0, abs(l64.item()))
    close(x.grad, x64.grad, dtype)


def test_loss_edge_rows():
    """Rows with -inf logits (masked vocabulary), the type's lowest value and large spreads; one position per
    sequence (nothing counted: NaN, as torch's mean of nothing, and a zero gradient)."""
    from loopback_amd import lm_ops as ops
    x = rnd((1, 6, 4100), torch.bfloat16, 10)
    x[0, 0, 5:] = float("-inf")
    x[0, 1] = torch.finfo(torch.bfloat16).min
    x[0, 2, 7] = 3e38
    x[0, 3, :4096] = float("-inf")
    ids = torch.tensor([[0, 3, 9, 7, 4099, 1]], device=DEV)
    x.requires_grad_()
    loss = ops.next_token_loss(x, ids)
    loss.backward()
    ref = x.detach().float().requires_grad_()
    lr = F.cross_entropy(ref[0, :-1], ids[0, 1:])
    lr.backward()
    assert torch.allclose(loss, lr, rtol=1e-6)
    close(x.grad, ref.grad, torch.bfloat16)
    one = rnd((2, 1, 64), torch.bfloat16, 11).requires_grad_()
    loss = ops.next_token_loss(one, torch.zeros(2, 1, dtype=torch.int64, device=DEV))
    loss.backward()
    assert loss.isnan() and not one.grad.any()


@pytest.mark.parametrize("m,n,k", [(1, 8, 8), (63, 264, 40), (65, 256, 256), (700, 40, 520), (1600, 512, 264),
                                   (8200, 776, 768)])
def test_wgrad(m, n, k):
    """dy^T x: one and several runs of tokens, remainders of a step, a tile and a run. Half a step of the result, and of
    fp32 sums over m products 1e-5 of the RMS per 16384 tokens (a fraction of it here)."""
    from loopback_amd import lm_ops as ops
    print(f"case wgrad {m}x{n}x{k} in {ops.LIB.llm_wgrad_splits(m, n, k)} runs", flush=True)
    dy, x = rnd((m, n), torch.bfloat16, m), rnd((m, k), torch.bfloat16, n)
    close(ops.wgrad(dy, x), dy.double().t() @ x.double(), torch.bfloat16)


def test_linear_module():
    """The layer's output and input gradient are torch's bits, its weight gradient at most as far from fp64 as torch's;
    second derivatives are torch's; few tokens stay on torch's product."""
    from loopback_amd import lm, lm_ops as ops
    torch.manual_seed(1)
    lin = lm.Linear(256, 512, bias=False).to(DEV, torch.bfloat16)
    x, g = rnd((2, 4100, 256), torch.bfloat16, 15).requires_grad_(), rnd((2, 4100, 512), torch.bfloat16, 16)
    y = lin(x)
    assert type(y.grad_fn).__name__ == "_LinearBackward"
    dx, dw = torch.autograd.grad(y, (x, lin.weight), g)
    yr = F.linear(x, lin.weight)
    dxr, dwr = torch.autograd.grad(yr, (x, lin.weight), g)
    exact = g.double().view(-1, 512).t() @ x.detach().double().view(-1, 256)
    assert torch.equal(y, yr) and torch.equal(dx, dxr)
    assert (dw.double() - exact).norm() <= 1.01 * (dwr.double() - exact).norm()
    d1, = torch.autograd.grad(lin(x), x, g, create_graph=True)
    second, = torch.autograd.grad(d1.float().pow(2).sum(), lin.weight)
    d1, = torch.autograd.grad(F.linear(x, lin.weight), x, g, create_graph=True)
    ref, = torch.autograd.grad(d1.float().pow(2).sum(), lin.weight)
    assert (second - ref).float().norm() <= 1e-2 * ref.float().norm()
    assert type(lin(x[:, :10]).grad_fn).__name__ != "_LinearBackward"


def test_what_stays_torch():
    """Second derivatives are torch's; a hooked norm is called as a module; forward-mode, vmap and fp32 calls take
    torch's operations."""
    from loopback_amd import lm, lm_ops as ops
    x, w = rnd((5, 64), torch.bfloat16, 12).requires_grad_(), rnd((64,), torch.bfloat16, 13).requires_grad_()
    gu = rnd((5, 64), torch.bfloat16, 14).requires_grad_()

    def second(fn, *inputs):
        out = fn(*inputs)
        g = torch.autograd.grad(out, inputs, torch.ones_like(out), create_graph=True)
        return torch.autograd.grad(sum(t.float().pow(2).sum() for t in g), inputs)

    pairs = [(second(lambda a, b: ops.add_rms_norm(a, None, b, 1e-6)[1], x, w),
              second(lambda a, b: F.rms_norm(a, (64,), b, 1e-6), x, w)),
             (second(ops.swiglu, gu), second(ops._swiglu_torch, gu))]
    for got, ref in pairs:
        for a, b in zip(got, ref):
            assert (a - b).float().norm() <= 2e-2 * b.float().norm()
    block = lm.Block(lm.LMConfig(hidden_size=64, num_heads=4)).to(DEV, torch.bfloat16)
    seen = []
    y = block(x[None])
    block.mlp_norm.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    assert torch.allclose(block(x[None]).float(), y.float(), atol=2e-2) and seen == [torch.Size([1, 5, 64])]
    y, dy = torch.func.jvp(ops.swiglu, (gu.detach(),), (torch.ones_like(gu),))
    assert torch.equal(y, ops._swiglu_torch(gu.detach())) and dy.shape == y.shape
    assert torch.func.vmap(ops.swiglu)(gu.detach()[None]).shape == (1, 5, 32)
    assert not ops.native(x.detach().float())


def test_only_on_the_current_gpu(monkeypatch):
    """Tensors of a GPU that is not the current one stay on torch: the default stream is the current GPU's."""
    from loopback_amd import lm_ops as ops
    x = rnd((2, 16), torch.bfloat16, 30)
    assert ops.native(x)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: x.device.index + 1)
    assert not ops.native(x)


def test_norm_without_eps():
    """RMSNorm's own default, eps None (the type's epsilon), is torch's operation."""
    from loopback_amd import lm
    x, norm = rnd((3, 64), torch.bfloat16, 31), lm.RMSNorm(64).to(DEV, torch.bfloat16)
    ref = F.rms_norm(x, (64,), norm.weight, None)
    assert torch.equal(norm(x), ref) and torch.equal(lm.add_norm(norm, x)[1], ref)


def test_dispatch_modes_see_torch_operations():
    """make_fx records the operations of a norm, SwiGLU and the loss: its graph gives their results on other inputs (to
    a few roundings of bf16, half a step 2^-9 to 2^-8 each)."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from loopback_amd import lm, lm_ops as ops
    norm = lm.RMSNorm(64, eps=1e-6).to(DEV, torch.bfloat16).requires_grad_(False)
    ids = torch.arange(6, device=DEV).view(2, 3)

    def fn(x):
        y = lm.add_norm(norm, x, x)[1]
        return ops.swiglu(y), ops.next_token_loss(y, ids)

    graph = make_fx(fn)(rnd((2, 3, 64), torch.bfloat16, 32))
    x = rnd((2, 3, 64), torch.bfloat16, 33)
    for got, ref in zip(graph(x), fn(x)):
        assert (got.float() - ref.float()).norm() <= 2e-2 * ref.float().norm()


@pytest.mark.parametrize("scale,vocab", [(0.5, 32000), (4.0, 32000), (20.0, 4096), (1.0, 33)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fast_exponential_costs_no_accuracy(scale, vocab, dtype):
    """The loss, its gradient and SwiGLU with its gradient are no further from 64 bits than torch's fp32 forms: the loss
    to an fp32 rounding (2^-24 of it), gradients to a ten-thousandth of the distance their 16-bit rounding leaves."""
    from loopback_amd import lm_ops as ops
    print(f"case fast exponential {scale} {vocab} {dtype}", flush=True)
    ids = torch.randint(0, vocab, (2, 128), generator=torch.Generator().manual_seed(40)).to(DEV)
    x, gu = scale * rnd((2, 128, vocab), dtype, 41), scale * rnd((256, 1024), dtype, 42)
    da, err = rnd((256, 512), dtype, 43), lambda a, b: ((a.double() - b).norm() / b.norm()).item()

    def run(loss, swiglu, cast):
        a, b = cast(x.detach()).requires_grad_(), cast(gu.detach()).requires_grad_()
        lo, act = loss(a), swiglu(b)
        return [lo.detach(), torch.autograd.grad(lo, a)[0], act.detach(), torch.autograd.grad(act, b, cast(da))[0]]

    exact = run(lambda a: F.cross_entropy(a[:, :-1].reshape(-1, vocab), ids[:, 1:].reshape(-1)), ops._swiglu_torch,
                torch.Tensor.double)
    got = run(lambda a: ops._NextTokenLoss.apply(a, ids), ops._SwiGLU.apply, lambda t: t)
    ref = run(ops._loss_torch(ids), ops._swiglu_torch, lambda t: t)
    for i, (a, b, e) in enumerate(zip(got, ref, exact)):
        assert err(a, e) <= err(b, e) * (1 + 1e-4) + (2.0 ** -24 if i == 0 else 0.0), i
