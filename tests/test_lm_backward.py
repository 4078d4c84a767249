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
