"""The launches chosen for few tokens (smaller write tiles, read tiles and backward tiles, the update gradient's one-row
lanes) against the ones for many: every token's values come from the same sums in the same order, so a token's final
state and gradients are bitwise the same alone, in a few and among 16 thousand (the query gradient, a sum over tokens
in tiles, is compared with the exact chain by every chain test). Sizes straddle each rule: a tile and its remainder,
the last count of the small launches and the first of the large ones."""
import pytest
import torch

from gpu_helpers import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,dtype", [(256, torch.bfloat16), (264, torch.bfloat16), (256, torch.float16),
                                     (768, torch.float32), (264, torch.float32), (2048, torch.bfloat16),
                                     (3072, torch.float32)])
@pytest.mark.parametrize("per_read", [False, True])
def test_tokens_do_not_depend_on_the_count(monkeypatch, d, dtype, per_read):
    from loopback_amd.chain import ChainConfig, make_inputs, run_chain
    if per_read:
        monkeypatch.setenv("LOOP_DATTN_GRAD_ROUNDING", "per_read")
    T = 16384 + 17
    cfg = ChainConfig(f"count-d{d}", d, 2, 3, 1, T, dtype, True, q_std=0.5)
    print(f"case token counts d{d} {dtype} per_read={per_read}", flush=True)
    h0, D, Q, G = make_inputs(cfg, DEV)
    h, _, g = run_chain(cfg, h0, D, Q, G, "scores")
    for n in (1, 15, 17, 4097, 8191, 16383):
        few = ChainConfig(f"count-d{d}-t{n}", d, 2, 3, 1, n, dtype, True, q_std=0.5)
        cut = lambda x: x[:, T - n:].contiguous()
        hf, _, gf = run_chain(few, cut(h0), [cut(x) for x in D], Q, cut(G), "scores")
        assert torch.equal(hf, cut(h)) and torch.equal(gf["h0"], cut(g["h0"])), n
        assert all(torch.equal(a, cut(b)) for a, b in zip(gf["D"], g["D"])), n
