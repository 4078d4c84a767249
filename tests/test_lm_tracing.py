"""The language model's layers under what has to see torch operations: the kernels leave those calls to torch before
they ask anything of the GPU or branch on a value."""
import pytest
import torch

from loopback_amd import lm

CFG = lm.LMConfig(hidden_size=128, num_heads=2, hidden_ratio=2)


def _on_gpu_bf16(make):
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device("cuda"):
            return make()
    finally:
        torch.set_default_dtype(torch.float32)


@pytest.mark.parametrize("make", [lambda: lm.SwiGLU(CFG), lambda: lm.RMSNorm(128, eps=1e-6), lambda: lm.Block(CFG).mlp_norm])
def test_fake_gpu_tensors(make):
    """16-bit layers over fake GPU tensors (shapes without data or a device), eager and compiled in one graph."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    graphs = []

    def backend(gm, inputs):
        graphs.append(gm)
        return gm.forward

    with FakeTensorMode():
        layer = _on_gpu_bf16(make)
        x = torch.empty(2, 8, 128, device="cuda", dtype=torch.bfloat16)
        y = layer(x)
        assert y.shape == x.shape and y.device == x.device
        torch._dynamo.reset()
        assert torch.compile(layer, backend=backend, fullgraph=True)(x).shape == x.shape
    assert len(graphs) == 1


@pytest.mark.gpu
def test_compiled_block_is_one_graph():
    """torch.compile of a bf16 block on the GPU: one graph, the eager torch form's results (a few bf16 roundings)."""
    block = lm.Block(CFG).to("cuda", torch.bfloat16)
    x = torch.randn(2, 8, 128, generator=torch.Generator().manual_seed(1)).to("cuda", torch.bfloat16)
    print("case compiled block", flush=True)
    torch._dynamo.reset()
    with torch.no_grad():
        got, ref = torch.compile(block, backend="eager", fullgraph=True)(x), block(x)
    assert (got.float() - ref.float()).norm() <= 2e-2 * ref.float().norm()


def test_layers_are_torch_modules():
    """What finds layers by their type finds the model's: its linear layers and norms are torch's own classes, dynamic
    quantization replaces them, torch.fx keeps them as leaves (with SwiGLU's operations between), and a SwiGLU and a
    norm can be scripted. Each gives the eager results."""
    from torch import nn
    block = lm.Block(CFG)
    assert [type(m) for m in block.modules() if isinstance(m, (nn.Linear, nn.RMSNorm))] == \
        [nn.RMSNorm, nn.Linear, nn.Linear, nn.RMSNorm, nn.Linear, nn.Linear]
    assert type(lm.LoopbackLM(lm.LMConfig(hidden_size=64, num_heads=2, vocab_size=32)).norm) is nn.RMSNorm
    x = torch.randn(2, 8, 128)

    class AttentionLeaf(torch.fx.Tracer):
        def is_leaf_module(self, m, name):
            return isinstance(m, lm.Attention) or super().is_leaf_module(m, name)

    tracer = AttentionLeaf()
    graph = tracer.trace(block)
    assert [n.target for n in graph.nodes if n.op == "call_module"] == \
        ["attn_norm", "attn", "mlp_norm", "mlp.gate_up", "mlp.down"]
    ref = block(x)
    assert torch.equal(torch.fx.GraphModule(tracer.root, graph)(x), ref)
    assert torch.equal(torch.fx.symbolic_trace(lm.RMSNorm(128, eps=1e-6))(x), lm.RMSNorm(128, eps=1e-6)(x))
    assert torch.allclose(torch.jit.script(block.mlp)(x), block.mlp(x), atol=1e-6)
    assert torch.allclose(torch.jit.script(block.mlp_norm)(x), block.mlp_norm(x), atol=1e-6)
    quantized = torch.ao.quantization.quantize_dynamic(block, {nn.Linear}, dtype=torch.qint8)
    assert not any(isinstance(m, nn.Linear) for m in quantized.modules())
    assert (quantized(x) - ref).norm() <= 5e-2 * ref.norm()   # 8-bit weights and activations


def test_a_hooked_linear_layer_is_called(monkeypatch):
    """A linear layer whose call is hooked, or that has a bias, is called as a module where the kernel would take it."""
    from torch import nn
    monkeypatch.setattr(lm.ops, "linear_native", lambda x, w: True)
    x = torch.randn(2, 16)
    for bias, hooked, calls in ((False, False, 0), (False, True, 1), (True, False, 0)):
        layer, seen = nn.Linear(16, 8, bias=bias), []
        taken = []
        monkeypatch.setattr(lm.ops, "linear", lambda x, w: taken.append(1) or torch.nn.functional.linear(x, w))
        if hooked:
            layer.register_forward_hook(lambda m, i, o: seen.append(1))
        assert torch.equal(lm.linear(layer, x), layer.forward(x))
        assert len(seen) == calls and bool(taken) == (not hooked and not bias)


def test_attention_operands_are_checked(monkeypatch):
    """A projection whose width is not the heads' is refused, as the torch form refuses its view, and tables the kernels
    do not index (another width, type or order of halves) go to the torch form."""
    taken = []
    monkeypatch.setattr(lm.ops, "attention_native", lambda qkv, dh: True)
    monkeypatch.setattr(lm.ops, "rotary_attention", lambda qkv, cos, sin, h, again: taken.append(1) or again(qkv))
    x = torch.randn(1, 5, 128)
    attn = lm.Attention(CFG)
    y = attn(x)
    assert taken == [1]
    attn.qkv = torch.nn.Linear(128, 2 * 128, bias=False)
    with pytest.raises(RuntimeError, match="shape"):
        attn(x)
    attn = lm.Attention(CFG)
    cos, sin = attn.rotary.tables(5, x.device, x.dtype)
    attn.rotary.tables = lambda *a: (cos.flip(-1), sin)
    taken.clear()
    assert attn(x).shape == y.shape and not taken
    ok = lambda c, s, heads=2, width=384: lm.ops.tables_native(torch.empty(1, 5, width), c, s, heads)
    assert ok(cos, sin)
    assert not any((ok(cos, sin, 3), ok(cos, sin, 2, 256), ok(cos.double(), sin), ok(cos, sin[:4]), ok(cos[:, :32], sin),
                    ok(cos, sin.t().contiguous().t())))
