"""The unaligned-row kernels (8 <= d <= 8192, any width and alignment) at the edges of their layouts: the narrowest
row, one element past and short of a vector, of a wave's 512 and 2048 elements, of the widest row, several waves per
row; two and 64 sources (addresses by value), 65 and 300 (device arrays, with fewer rows per workgroup)."""
import pytest
import torch

from gpu_helpers import DEV, err_rms, make
from test_gpu_read import compare, run_hip, run_oracle
from test_gpu_stack import check_chain, hip_chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,t,d,n", [(1, 70, 8, 3), (1, 70, 9, 2), (3, 11, 63, 64), (2, 9, 511, 5), (2, 9, 513, 6),
                                     (1, 13, 2047, 4), (1, 13, 2049, 7), (1, 3, 8191, 5), (1, 6, 40, 300),
                                     (1, 5, 1001, 65), (1, 2, 4097, 65)])
def test_list_read_at_layout_edges(b, t, d, n):
    """Forward and every gradient within 1e-5 x RMS of the exact read, the bar of every fp32 read."""
    args = make(b, t, d, n, torch.float32, seed=7 * n + d)
    print(f"case unaligned rows b{b} t{t} d{d} n{n}", flush=True)
    e64 = compare(run_hip(d, n, args, True), run_oracle(d, n, args, True, dtype=torch.float64), err_rms)
    assert max(e64.values()) <= 1e-5, e64


@pytest.mark.parametrize("d", [9, 1001, 4099])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_chain_at_layout_edges(d, dtype):
    """A stacked chain (the write, the update gradients, the blends' sum) to the chain bars."""
    from loopback_amd.chain import ChainConfig
    cfg = ChainConfig(f"rows-d{d}", d, 2, 3, 1, 67, dtype, True, q_std=0.5)
    print(f"case unaligned chain d{d} {dtype}", flush=True)
    h, g = hip_chain(cfg, "scores")
    check_chain(h, g, cfg)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [3, 9, 130, 1001])
def test_write_stores_the_scale_of_rstd(dtype, d):
    """V = h - x as torch subtracts, R bitwise the scale kernel's (one summation order for both)."""
    from loopback_amd import fused_dattn as FD
    g = torch.Generator().manual_seed(d)
    h, x = (torch.randn(1, 37, d, generator=g).to(dtype).to(DEV) for _ in range(2))
    stack = FD.DattnStack(2, (1, 37, d), dtype, DEV)
    print(f"case unaligned write d{d} {dtype}", flush=True)
    with torch.no_grad():
        v = stack.write(0, h, x)
        r = FD.rstd(v, stack.eps)
    torch.cuda.synchronize()
    assert torch.equal(v, h - x) and torch.equal(stack.R[0], r.view_as(stack.R[0]))


def read_errors(d, n, t=300):
    """The 2-norm errors from 64 bits of an fp32 read and of a model of it in fp32 torch operations that adds one
    weight per source, each addition rounded once."""
    from loopback_amd import fused_dattn as FD
    g = torch.Generator().manual_seed(d + n)
    base, q = torch.randn(1, t, d, generator=g), 0.3 * torch.randn(d, generator=g)
    vs = [torch.randn(1, t, d, generator=g) for _ in range(n)]
    c0 = torch.rand(n, generator=g) * 0.9 + 0.1
    cbar = c0 + 0.2 * torch.randn(1, t, n, generator=g)
    rs = [FD.rstd_ref(v, 1e-6) for v in vs]
    dev = lambda ts: [x.to(DEV) for x in ts]
    with torch.no_grad():
        out, _ = FD.FusedDattnRead.apply(*dev((q, base, cbar, c0, *vs, *rs)))

    def weights(dt):
        z = torch.stack([(v.to(dt) @ q.to(dt)) * r.to(dt)[..., 0] for v, r in zip(vs, rs)], -1) / d ** 0.5
        lc, c = c0.to(dt).log(), c0.to(dt)
        return c + c.sum() * (torch.softmax(z + lc, -1) - torch.softmax(lc, -1)) - cbar.to(dt)

    exact, model, w64, w32 = base.double(), base, weights(torch.float64), weights(torch.float32)
    for i, v in enumerate(vs):
        exact = exact + w64[..., i:i + 1] * v.double()
        model = (model.double() + w32[..., i:i + 1].double() * v.double()).float()
    return (out.cpu().double() - exact).norm().item(), (model.double() - exact).norm().item()


@pytest.mark.parametrize("d,n", [(333, 2), (1001, 8), (1001, 24), (768, 72), (2049, 64), (4099, 12)])
def test_read_error_of_one_weight_per_source(d, n):
    """fp32 reads whose softmax is formed as the sources stream (their fixed and softmax shares summed apart) are no
    further from 64 bits than one weight per source in fp32 (0.5 to 0.9 of it; without compensated sums 1.0 to 1.8)."""
    got, model = read_errors(d, n)
    print(f"case read error d{d} n{n}: {got:.3e}, one weight per source {model:.3e}, ratio {got / model:.3f}", flush=True)
    assert got <= model


def test_infinite_base_element():
    """An infinite element of the base stays infinite, and alone (the compensated sums do not see it)."""
    from loopback_amd import fused_dattn as FD
    g = torch.Generator().manual_seed(3)
    base, q, cbar = torch.randn(1, 5, 333, generator=g), torch.randn(333, generator=g), torch.rand(1, 5, 6, generator=g)
    base[0, 2, 331] = float("inf")
    vs = [torch.randn(1, 5, 333, generator=g).to(DEV) for _ in range(6)]
    rs = [FD.rstd(v, 1e-6) for v in vs]
    with torch.no_grad():
        out, _ = FD.FusedDattnRead.apply(q.to(DEV), base.to(DEV), cbar.to(DEV), torch.ones(6, device=DEV), *vs, *rs)
    out = out.cpu()
    assert out[0, 2, 331] == float("inf") and out.isfinite().sum() == out.numel() - 1


@pytest.mark.parametrize("d,n", [(2000, 900), (2000, 1000), (1500, 1024), (8192, 1024)])
def test_many_sources_of_wide_fp32_rows(d, n):
    """The query and a workgroup's per-source scalars in LDS at its bound (62192 bytes), and past it with half the rows
    per workgroup: the read of one weight per source."""
    got, model = read_errors(d, n, 5)
    print(f"case wide rows d{d} n{n}: {got:.3e}, one weight per source {model:.3e}", flush=True)
    assert got <= model
