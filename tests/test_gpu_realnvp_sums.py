"""Rounding of the RealNVP passes' sums over the hidden features, against FP64.

One layer whose scale head is zero (s = 0) and whose transformed inputs are zero
returns the shift head's sum alone: y = W2 relu(W1 c + b1). Its error is held to
that of the same sum in FP32 over S strided chains that are added pairwise (S =
256 / (4 ceil(n_trans / 4)) rounded down to a power of two, at most 64): with k
features a chain the variance of its rounding error is (k + 1) / 2 + log2 S
units of one addition's. The passes' chains of 4 or 8 features and their pairs
stay below it at every width here (largest ratio of the rms errors expected:
1.02), a chain through all features is at 2 to 4 times. 1.1 leaves the room of the
sampled rms. Reference: src/flowMC/resource/model/nf_model/realNVP.py:62-99.
"""

import numpy as np
import pytest
import torch

from flowmc_amd import random as fr
from flowmc_amd.resource.model.nf_model.realNVP import RealNVP

pytestmark = pytest.mark.gpu

ROWS = 2000  # rows whose sums are followed on the CPU


def fma(a, b, c):
    """a b + c rounded to FP32 once (the FP64 product is exact)."""
    return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(np.float32)


# n: a tile shared by a workgroup, 16 and 32 samples a wavefront
@pytest.mark.parametrize("n", [2000, 24000, 40000])
@pytest.mark.parametrize("d,h", [(32, 256), (32, 1000), (5, 64), (64, 128), (130, 64)])
def test_hidden_sums(gpu, d, h, n):
    g = torch.Generator().manual_seed(h + d)
    half = d // 2
    W1, b1 = torch.randn(h, d, generator=g) / d ** 0.5, torch.randn(h, generator=g) * 0.1
    W2 = torch.randn(d, h, generator=g) / h ** 0.5
    zero = [torch.zeros(h, d), torch.zeros(h), torch.zeros(d, h), torch.zeros(d)]
    stats = [torch.zeros(d), torch.eye(d), torch.zeros(d), torch.eye(d)]
    theta = torch.cat([p.reshape(-1) for p in zero + [W1, b1, W2, torch.zeros(d)] + stats])
    m = RealNVP(d, 1, h, fr.PRNGKey(0), _theta=theta)
    cond, trans = (list(range(half)), list(range(half, d)))  # layer 0 conditions on the first half
    x = torch.zeros(n, d)
    x[:, cond] = torch.randn(n, half, generator=g)
    y, _ = m.forward(x.cuda())
    got = y[:ROWS].cpu()[:, trans].numpy().astype(np.float64)

    xc, w1, w2 = x[:ROWS, cond].numpy(), W1[:, cond].numpy(), W2[trans].numpy()
    hid = np.broadcast_to(b1.numpy(), (ROWS, h)).astype(np.float32)
    for k in range(half):
        hid = fma(xc[:, k:k + 1], w1[None, :, k], hid)
    hid = np.maximum(hid, np.float32(0))
    exact = hid.astype(np.float64) @ w2.T.astype(np.float64)
    S = 1
    while S < 64 and 4 * ((len(trans) + 3) // 4) * S * 2 <= 256:
        S *= 2
    acc = np.zeros((S, ROWS, len(trans)), np.float32)
    for j in range(h):
        acc[j % S] = fma(hid[:, j:j + 1], w2[None, :, j], acc[j % S])
    while len(acc) > 1:
        acc = acc[:len(acc) // 2] + acc[len(acc) // 2:]

    def rms(v):
        return float(np.sqrt(np.mean((v - exact) ** 2)))

    assert rms(got) <= 1.1 * rms(acc[0].astype(np.float64))


def _close(a, b):
    return float(((a.detach().cpu().double() - b).abs() / (1 + b.abs())).max()) <= 2e-4


# the batches around which the pass changes (hidden 20, two blocks: 512 tiles of
# 16 samples shared by a workgroup each, then a wavefront each), against the
# FP64 oracle: FP32 products of up to a few hundred terms a layer, errors
# growing a few-fold over the layers
@pytest.mark.parametrize("n", [8192, 8193, 20000])
@pytest.mark.parametrize("d", [5, 33, 70, 150])
def test_passes_around_the_rule(gpu, d, n):
    from oracle import realnvp as R

    p = R.init_params(d, 2, 20, seed=d, scale=0.5, out_scale=1.0 / 20 ** 0.5)
    p["data_mean"] = torch.linspace(-0.5, 0.5, d, dtype=torch.float64)
    p["data_cov"] = torch.diag(torch.linspace(0.5, 1.5, d, dtype=torch.float64))
    theta = R.to_flat(p).float()
    m, p = RealNVP(d, 2, 20, fr.PRNGKey(0), _theta=theta), R.from_flat(theta.double(), d, 2, 20)
    x = torch.randn(n, d, generator=torch.Generator().manual_seed(n + d))
    for got, want in ((m.forward(x.cuda()), R.forward(p, x.double())), (m.inverse(x.cuda()), R.inverse(p, x.double()))):
        assert _close(got[0], want[0]) and _close(got[1], want[1])
    assert _close(m.log_prob(x.cuda()), R.log_prob(p, x.double()))


@pytest.mark.parametrize("d,trans", [(40, 1), (40, 39), (40, 40), (40, 0), (130, 120), (130, 5)])
def test_uneven_masks_a_wavefront_each(gpu, d, trans):
    from flowmc_amd.resource.model.nf_model.realNVP import AffineCoupling
    from oracle import realnvp as R

    mask = torch.zeros(d)
    mask[torch.randperm(d, generator=torch.Generator().manual_seed(trans))[:trans]] = 1.0  # 1 = transformed
    layer = AffineCoupling(d, 20, mask, fr.PRNGKey(3), 0.5, scale=0.5)
    x = torch.randn(9001, d, generator=torch.Generator().manual_seed(d))
    y, ld = layer.forward(x.cuda())
    lp = R.from_flat(layer.theta.cpu().double(), d, 1, 20)["layers"][0]
    ry, rld = R.affine_coupling(lp, x.double(), 1 - mask.double(), dt=0.5)
    assert _close(y, ry) and _close(ld, rld)
