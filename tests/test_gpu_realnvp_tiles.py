"""RealNVP passes at the edges of their tiles and of the rules that choose
them: batches of one sample, one tile, one more than a tile, and sizes that
take each of the pass kernels; dims and masks that leave one, two, four and
more blocks of 16 on a side. Against the FP64 oracle on the FP32-rounded
parameters, within 2e-4 * (1 + |ref|) (FP32 products of up to a few hundred
terms per layer, errors growing a few-fold over the layers)."""

import pytest
import torch

from flowmc_amd import random as fr
from flowmc_amd.resource.model.nf_model.realNVP import AffineCoupling, RealNVP
from oracle import realnvp as R

pytestmark = pytest.mark.gpu


def make(d, L, h, seed=0):
    p = R.init_params(d, L, h, seed=seed, scale=0.5, out_scale=1.0 / h ** 0.5)
    p["data_mean"] = torch.linspace(-0.5, 0.5, d, dtype=torch.float64)
    p["data_cov"] = torch.diag(torch.linspace(0.5, 1.5, d, dtype=torch.float64))
    theta = R.to_flat(p).float()
    return RealNVP(d, L, h, fr.PRNGKey(0), _theta=theta), R.from_flat(theta.double(), d, L, h)


def close(a, b, tol=2e-4):
    return float(((a.detach().cpu().double() - b).abs() / (1 + b.abs())).max()) <= tol


# hidden 20 is two blocks: a shared tile up to 3200 samples, then 16 and (past 32,768) 32 samples a wave
@pytest.mark.parametrize("n", [1, 15, 16, 17, 3201, 5000, 32769])
@pytest.mark.parametrize("d", [2, 5, 33])
def test_passes_at_tile_edges(gpu, n, d):
    m, p = make(d, 2, 20)
    x = torch.randn(n, d, generator=torch.Generator().manual_seed(n + d))
    y, ld = m.forward(x.cuda())
    ry, rld = R.forward(p, x.double())
    assert close(y, ry) and close(ld, rld)
    xi, li = m.inverse(x.cuda())
    rxi, rli = R.inverse(p, x.double())
    assert close(xi, rxi) and close(li, rli)
    assert close(m.log_prob(x.cuda()), R.log_prob(p, x.double()))


@pytest.mark.parametrize("d,n", [(70, 40), (70, 5000), (150, 40), (150, 5000), (150, 33000), (300, 40)])
def test_passes_with_many_blocks(gpu, d, n):
    m, p = make(d, 2, 20, seed=1)
    x = torch.randn(n, d, generator=torch.Generator().manual_seed(d))
    y, ld = m.forward(x.cuda())
    ry, rld = R.forward(p, x.double())
    assert close(y, ry) and close(ld, rld)
    assert close(m.inverse(x.cuda())[0], R.inverse(p, x.double())[0])


@pytest.mark.parametrize("n", [40, 5000, 33000])
@pytest.mark.parametrize("d,trans", [(40, 1), (40, 39), (40, 40), (40, 0), (130, 120), (130, 5)])
def test_coupling_with_uneven_masks(gpu, n, d, trans):
    mask = torch.zeros(d)
    mask[torch.randperm(d, generator=torch.Generator().manual_seed(trans))[:trans]] = 1.0  # 1 = transformed
    layer = AffineCoupling(d, 20, mask, fr.PRNGKey(3), 0.5, scale=0.5)
    x = torch.randn(n, d, generator=torch.Generator().manual_seed(n))
    y, ld = layer.forward(x.cuda())
    lp = R.from_flat(layer.theta.cpu().double(), d, 1, 20)["layers"][0]
    ry, rld = R.affine_coupling(lp, x.double(), 1 - mask.double(), dt=0.5)
    assert close(y, ry) and close(ld, rld)
    xr, li = layer.inverse(y)
    assert close(xr, x.double()) and close(li, -ld.cpu().double())


def decided(p, x):
    """Rows whose hidden pre-activations all lie further than FP32 rounding
    from the ReLU's kink (in FP64): on the others either side is right, and an
    input gradient jumps between the two."""
    d, L = x.shape[1], len(p["layers"])
    z = (x.double() - p["data_mean"]) / torch.sqrt(torch.diagonal(p["data_cov"]))
    near = torch.full((x.shape[0],), 1.0, dtype=torch.float64)
    for l in range(L):
        lp, mk = p["layers"][l], R.mask(d, l, torch.float64)
        for t in "st":
            near = torch.minimum(near, ((z * mk) @ lp[f"W{t}1"].T + lp[f"b{t}1"]).abs().amin(1))
        z, _ = R.affine_coupling(lp, z, mk, 1.0)
    return near > 1e-6


# tiles of 16, 32 and 48 samples (one group of 16 up to 4096 samples, two up
# to 8192), masks in one to ten blocks, hidden layers of one block, a ragged
# number and more than the eight waves share. Gradients are sums over the
# batch of FP32 products: within 2e-3 of the largest entry, as for the
# single-tile sizes (a ReLU mask decided differently in FP64 moves an entry by
# one sample's share of a few thousand).
@pytest.mark.parametrize("d,h,n", [(2, 8, 1), (5, 20, 16), (5, 64, 17), (5, 20, 4097), (6, 70, 8193), (33, 20, 40),
                                   (33, 20, 4097), (40, 100, 8200), (70, 20, 50), (150, 20, 40), (300, 20, 20)])
def test_adjoint_at_tile_edges(gpu, d, h, n):
    m, p = make(d, 3, h, seed=2)
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, d, generator=g)
    w = torch.rand(n, generator=g) + 0.5
    gt, gx = m.grad_log_prob_sum(x.cuda(), w.cuda())
    theta = R.to_flat(p).clone().requires_grad_(True)
    xr = x.double().clone().requires_grad_(True)
    obj = (w.double() * R.log_prob(R.from_flat(theta, d, 3, h), xr)).sum()
    rg, rgx = torch.autograd.grad(obj, [theta, xr])
    k = 3 * 2 * (2 * h * d + h + d)
    assert float((gt.cpu().double()[:k] - rg[:k]).abs().max()) <= 2e-3 * float(rg[:k].abs().max())
    ok = decided(p, x)
    assert int((~ok).sum()) <= 1 + n // 500
    assert float((gx.cpu().double() - rgx)[ok].abs().max()) <= 2e-3 * float(rgx.abs().max())
    assert float(gt.cpu()[k:].abs().max()) == 0.0
