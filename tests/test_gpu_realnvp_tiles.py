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
