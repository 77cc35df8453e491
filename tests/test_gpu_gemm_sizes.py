"""The GEMM kernels at the sizes where their tiles, remainders and dispatch
rules change, against 64-bit products of the same values."""
import pytest
import torch

pytestmark = pytest.mark.gpu

dev = "cuda"


def say(*a):
    print("[case]", *a, flush=True)


# K off and on the matrix kernels' grid (20, 40: the SIMT kernel); rows and
# channels around the 16-, 32- and 64-wide tiles, channel counts not a
# multiple of 4 (element-wise stores), more row tiles than CUs
@pytest.mark.parametrize("n,k,n_out", [(1, 32, 8), (16, 64, 16), (17, 96, 17), (16, 32, 66),
                                       (17, 32, 33), (33, 512, 64), (64, 96, 130), (65, 256, 1000),
                                       (5000, 32, 8), (2100, 64, 640), (40, 20, 48), (129, 40, 70)])
def test_f32_linear_tile_edges(n, k, n_out):
    from spider_moe_amd import ForgeConfig
    from spider_moe_amd.forge import ForgeGEMM
    say("f32 linear", n, k, n_out)
    g = torch.Generator().manual_seed(n * 7 + k + n_out)
    x = torch.randn(n, k, generator=g)
    w = torch.randn(n_out, k, generator=g)
    b = torch.randn(n_out, generator=g)
    y = ForgeGEMM(ForgeConfig()).linear(x.to(dev), w.to(dev), b.to(dev)).cpu().double()
    ref = x.double() @ w.double().t() + b.double()
    # k products and k + 1 sums in f32, in any order: each at most 2^-24 off,
    # relative to the sum of magnitudes
    bound = (2 * k + 2) * 2.0 ** -24 * (x.abs().double() @ w.abs().double().t() + b.abs().double())
    assert bool(((y - ref).abs() <= bound).all())


# experts with no rows, one row and partial tiles; top_k 1 leaves groups of
# about n / e rows: 4 and 16 (16-row tiles), 17 and 100 (32- and 64-row tiles)
@pytest.mark.parametrize("n,h,u,e,k", [(32, 64, 96, 8, 1), (128, 32, 64, 8, 1), (136, 64, 128, 8, 1),
                                       (400, 96, 160, 8, 2), (3000, 64, 320, 5, 2)])
def test_f32_grouped_tile_edges(n, h, u, e, k):
    from spider_moe_amd import sparse_expert_delta
    say("f32 grouped", n, h, u, e, k)
    g = torch.Generator().manual_seed(n + h + u)
    x = torch.randn(1, n, h, generator=g)
    idx = torch.randint(0, e - 1, (n, k), generator=g)  # the last expert stays empty ...
    idx[0, 0] = e - 1                                   # ... but for one row
    idx[1:, 0] = torch.where(idx[1:, 0] == 1, torch.zeros(()).long(), idx[1:, 0])  # expert 1: k > 1 only
    wt = torch.rand(n, k, generator=g) + 0.1
    wu, bu = torch.randn(e, u, h, generator=g) * h ** -0.5, torch.randn(e, u, generator=g)
    wd, bd = torch.randn(e, h, u, generator=g) * u ** -0.5, torch.randn(e, h, generator=g)
    y = sparse_expert_delta(x.to(dev), idx.view(1, n, k).to(dev), wt.view(1, n, k).to(dev), wu.to(dev),
                            bu.to(dev), wd.to(dev), bd.to(dev), num_experts=e, top_k=k).cpu().double()[0]
    ref = torch.zeros(n, h, dtype=torch.float64)
    mag = torch.zeros(n, h, dtype=torch.float64)
    for j in range(k):
        for x_ in range(e):
            r = (idx[:, j] == x_).nonzero().squeeze(-1)
            a = torch.nn.functional.gelu(x[0, r].double() @ wu[x_].double().t() + bu[x_].double())
            ref[r] += (a @ wd[x_].double().t() + bd[x_].double()) * wt[r, j:j + 1].double()
            mag[r] += (a.abs() @ wd[x_].abs().double().t() + bd[x_].abs().double()) * wt[r, j:j + 1].double()
    # the down product's sums as above; an up activation of size ~1 is off by
    # its own sums (h terms) and by erf's 1.5e-7, which the down weights carry on
    up_err = (2 * h + 2) * 2.0 ** -24 * 4 * h ** 0.5 + 2e-7
    bound = (2 * u + 8) * 2.0 ** -24 * mag + up_err * u ** 0.5 * wt.sum(-1, keepdim=True).double()
    assert bool(((y - ref).abs() <= bound).all())
