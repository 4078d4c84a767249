"""The backwards of the language model's kernel operations where they run torch's operations instead. On the CPU the
launches are left out: what is compared depends on the saved inputs alone."""
import pytest
import torch
import torch.nn.functional as F

from loopback_amd import lm, lm_ops as ops


@pytest.fixture
def no_launch(monkeypatch):
    monkeypatch.setattr(ops, "_run", lambda name, *args: None)
    monkeypatch.setattr(ops, "_stream", lambda t: 0)


def rnd(shape, seed, dtype=torch.bfloat16):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


@pytest.mark.parametrize("need_x,need_w", [(False, True), (True, False), (True, True)])
@pytest.mark.parametrize("add", [False, True])
def test_norm_second_derivatives(no_launch, need_x, need_w, add):
    """A norm's backward that is differentiated, with an input or a weight that needs no gradient: torch's."""
    x, w = rnd((5, 64), 1).requires_grad_(need_x), rnd((64,), 2).requires_grad_(need_w)
    a = rnd((5, 64), 3) if add else None
    g = rnd((5, 64), 4).requires_grad_()
    wanted = [t for t in (x, w) if t.requires_grad]

    def second(h, y):
        assert h.requires_grad == need_x
        first = torch.autograd.grad(y, wanted, g, create_graph=True)
        return first + torch.autograd.grad(sum(t.float().pow(2).sum() for t in first), [*wanted, g], allow_unused=True)

    h, y = ops.add_rms_norm(x, a, w, 1e-6)
    if add:
        h.data.copy_(x + a)
    hr = x if a is None else x + a
    got, ref = second(h, y), second(hr, F.rms_norm(hr, (64,), w, 1e-6))
    for p, q in zip(got, ref):
        assert (p is None) == (q is None) and (p is None or (p - q).float().norm() <= 2e-2 * q.float().norm() + 1e-6)


def test_norm_backward_forms_what_is_needed(monkeypatch):
    """A frozen gain gets no partial sums and no reduction, an input that needs no gradient none."""
    launches = []
    monkeypatch.setattr(ops, "_run", lambda name, *args: launches.append((name, args)))
    monkeypatch.setattr(ops, "_stream", lambda t: 0)
    for need_x, need_w in ((True, False), (False, True), (True, True)):
        x, w = rnd((5, 64), 1).requires_grad_(need_x), rnd((64,), 2).requires_grad_(need_w)
        y = ops.add_rms_norm(x, None, w, 1e-6)[1]
        launches.clear()
        y.backward(rnd((5, 64), 3))
        assert [n for n, _ in launches] == ["llm_rms_norm_bwd"] + ["llm_sum_rows"] * need_w
        assert (launches[0][1][5] is not None) == need_x and (launches[0][1][6] is not None) == need_w
    assert ops.LIB.llm_rms_norm_bwd(4096, 4096, 4096, 4096, None, None, None, 1, 64, 1, None) == -1   # neither


@pytest.mark.gpu
@pytest.mark.parametrize("rows,d", [(5, 64), (2049, 768), (9, 2048)])
def test_norm_gradients_one_at_a_time(rows, d):
    """Each gradient alone has the bits it has beside the other."""
    print(f"case norm gradients alone {rows}x{d}", flush=True)
    x, w, g = (rnd(s, k).cuda() for s, k in (((rows, d), 1), ((d,), 2), ((rows, d), 3)))
    got = {}
    for need in ((True, True), (True, False), (False, True)):
        a, b = x.clone().requires_grad_(need[0]), w.clone().requires_grad_(need[1])
        ops.add_rms_norm(a, None, b, 1e-6)[1].backward(g)
        got[need] = a.grad, b.grad
    both = got[True, True]
    assert torch.equal(got[True, False][0], both[0]) and got[True, False][1] is None
    assert torch.equal(got[False, True][1], both[1]) and got[False, True][0] is None


def _operations(monkeypatch):
    """name -> (the kernel operation, its torch form, the input it is differentiated by)."""
    monkeypatch.setattr(ops, "wgrad", lambda dy, x: pytest.fail("a weight gradient was launched"))
    w, u, ids = rnd((64,), 2), rnd((32, 64), 5), torch.arange(6).view(2, 3)
    cos, sin = lm.Rotary(64, 1e6).tables(3, "cpu", torch.bfloat16)
    attn = lm.Attention(lm.LMConfig(hidden_size=64, num_heads=1))
    return {"norm": (lambda x: ops.add_rms_norm(x, None, w, 1e-6)[1], lambda x: F.rms_norm(x, (64,), w, 1e-6),
                     rnd((5, 64), 1)),
            "swiglu": (ops._SwiGLU.apply, ops._swiglu_torch, rnd((5, 64), 1)),
            "loss": (lambda x: ops._NextTokenLoss.apply(x, ids), ops._loss_torch(ids), rnd((2, 3, 64), 1)),
            "linear": (lambda x: ops._Linear.apply(x, u), lambda x: F.linear(x, u), rnd((5, 64), 1)),
            "attention": (lambda x: ops.rotary_attention(x, cos, sin, 1, attn.attend), attn.attend, rnd((1, 3, 192), 1))}


@pytest.mark.parametrize("name", ["norm", "swiglu", "loss", "linear", "attention"])
@pytest.mark.parametrize("how", ["batched", "vmap", "mode"])
def test_watched_backwards(no_launch, monkeypatch, name, how):
    """Batched gradients, a vmap over the backward, and a dispatch mode around it: torch's operations."""
    fn, ref_fn, x = _operations(monkeypatch)[name]
    x.requires_grad_()
    y, yr = fn(x), ref_fn(x)
    gs = torch.stack([rnd(y.shape, k, y.dtype) for k in (7, 8)])

    def grads(out):
        if how == "batched":
            return torch.autograd.grad(out, x, gs, is_grads_batched=True)[0]
        if how == "vmap":
            return torch.func.vmap(lambda g: torch.autograd.grad(out, x, g, retain_graph=True)[0])(gs)
        from torch.utils.flop_counter import FlopCounterMode
        with FlopCounterMode(display=False):
            return torch.autograd.grad(out, x, gs[0])[0]

    assert torch.allclose(grads(y), grads(yr), rtol=1e-2, atol=1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["batched", "vmap", "mode", "plain"])
def test_watched_backwards_on_the_gpu(how):
    """The same through the engine's GPU thread, the forward by the kernels: torch's gradients, to a few roundings of
    bf16 (both round each result once, torch some intermediate ones too)."""
    print(f"case watched backward {how}", flush=True)
    dev = lambda *ts: [t.cuda() for t in ts]
    w, u, ids = dev(rnd((64,), 2), rnd((32, 64), 5), torch.arange(6).view(2, 3))
    for fn, ref_fn, shape in ((lambda x: ops.add_rms_norm(x, None, w, 1e-6)[1], lambda x: F.rms_norm(x, (64,), w, 1e-6), (5, 64)),
                              (ops._SwiGLU.apply, ops._swiglu_torch, (5, 64)),
                              (lambda x: ops._NextTokenLoss.apply(x, ids), ops._loss_torch(ids), (2, 3, 64)),
                              (lambda x: ops._Linear.apply(x, u), lambda x: F.linear(x, u), (5, 64))):
        x = rnd(shape, 1).cuda().requires_grad_()

        def grads(out):
            gs = torch.stack([rnd(out.shape, k, out.dtype) for k in (7, 8)]).cuda()
            if how == "batched":
                return torch.autograd.grad(out, x, gs, is_grads_batched=True)[0]
            if how == "vmap":
                return torch.func.vmap(lambda g: torch.autograd.grad(out, x, g, retain_graph=True)[0])(gs)
            if how == "plain":
                return torch.autograd.grad(out, x, gs[0])[0]
            from torch.utils.flop_counter import FlopCounterMode
            with FlopCounterMode(display=False):
                return torch.autograd.grad(out, x, gs[0])[0]

        got, ref = grads(fn(x)), grads(ref_fn(x))
        assert (got - ref).float().norm() <= 2e-2 * ref.float().norm()


def test_saved_tensors_with_other_strides():
    """What a saved-tensor hook gives back strided or unaligned reaches the kernels as contiguous aligned rows."""
    ctx = type("ctx", (), {})()
    x = rnd((4, 8), 1)
    ctx.saved_tensors = (x, x.t().contiguous().t(), torch.cat((x.new_zeros(1), x.flatten()))[1:].view(4, 8),
                         torch.ones(1)[0], x[:0])
    for got, t in zip(ops._saved(ctx), ctx.saved_tensors):
        assert torch.equal(got, t) and got.is_contiguous() and got.data_ptr() % 16 == 0
    assert ops._saved(ctx)[0] is x
    ctx.saved_tensors = (x,)
    assert ops._saved(ctx) is ctx.saved_tensors


@pytest.mark.gpu
def test_gradients_through_saved_tensor_hooks():
    """Hooks that transpose what is saved and give back transposed views: the gradients' bits without them."""
    w, ids = rnd((192,), 2).cuda().requires_grad_(), torch.arange(80).view(2, 40).cuda()
    cos, sin = lm.Rotary(64, 1e6).tables(40, torch.device("cuda", 0), torch.bfloat16)
    x = rnd((2, 40, 192), 1).cuda().requires_grad_()

    def grads():
        h, n = ops.add_rms_norm(x, None, w, 1e-6)
        a = ops.rotary_attention(n, cos, sin, 1, None)
        y = ops.add_rms_norm(ops.swiglu(h + n), a.repeat(1, 1, 3)[..., :96].contiguous(), w[:96].detach(), 1e-6)[1]
        return ops.next_token_loss(y, ids)

    print("case saved-tensor hooks", flush=True)
    ref = torch.autograd.grad(grads(), (x, w))
    turn = lambda t: t.transpose(0, -1).contiguous() if t.dim() > 1 else t
    with torch.autograd.graph.saved_tensors_hooks(turn, lambda t: t.transpose(0, -1) if t.dim() > 1 else t):
        loss = grads()
    for p, q in zip(torch.autograd.grad(loss, (x, w)), ref):
        assert torch.equal(p, q)


@pytest.mark.gpu
def test_block_gradients_with_a_graph():
    """A block fed plain activations, its parameters' gradients taken with a graph: those taken without."""
    block = lm.Block(lm.LMConfig(hidden_size=128, num_heads=2)).to("cuda", torch.bfloat16)
    x, g = rnd((2, 40, 128), 1).cuda(), rnd((2, 40, 128), 2).cuda()
    print("case block create_graph", flush=True)
    params = list(block.parameters())
    ref = torch.autograd.grad(block(x), params, g)
    got = torch.autograd.grad(block(x), params, g, create_graph=True)
    for p, q in zip(got, ref):
        assert (p - q).float().norm() <= 2e-2 * q.float().norm()


def test_weight_gradient_rule(monkeypatch):
    """Which linear layers record the split-token weight gradient: from 64 x 64 weights and 8192 tokens on, with at
    least five runs of tokens."""
    monkeypatch.setattr(ops, "native", lambda *ts: True)

    def takes(tokens, n, k):
        w = torch.empty(n, k, dtype=torch.bfloat16, requires_grad=True)
        return ops.linear_native(torch.empty(1, dtype=torch.bfloat16).expand(tokens, k), w)

    monkeypatch.setattr(ops, "_rows_ok", lambda *ts: True)
    assert [takes(*s) for s in ((8192, 64, 64), (8192, 4096, 768), (65536, 72, 2048), (12000, 3072, 1024))] == [True] * 4
    assert [takes(*s) for s in ((8191, 64, 64), (16384, 56, 512), (16384, 512, 16), (8192, 2048, 2048),
                                (8192, 4096, 1024), (16384, 5632, 1024), (16384, 68, 64))] == [False] * 7
