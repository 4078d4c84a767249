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
