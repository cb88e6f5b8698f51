"""Rounding of the RealNVP weight gradients' sums over the samples, against FP64.

One layer whose scale head is zero has y = x + t and, with g_logp = 1, the shift
head's output gradient -y, so that dW2[i][j] = -sum_m y[m][i] H[m][j] of
factors that are known to the bit. Its error is held to that of the same sum in
FP32 over tiles of 16 samples (a chain each), tile sums in 16 strided chunks of four
accumulators and the chunks one after the other. The adjoint sums 16 samples
a chain, a tile of one to three such chains, and the tiles in sixteen strided sums
that are added pairwise; one chain through 48 samples and a quarter of all tiles had
two to three times the error at the sizes here. 1.25 leaves the room of an rms over a few
hundred entries. Reference: src/flowMC/resource/model/nf_model/base.py:98-125.
"""

import numpy as np
import pytest
import torch

from flowmc_amd import random as fr
from flowmc_amd.resource.model.nf_model.realNVP import RealNVP

pytestmark = pytest.mark.gpu


def fma(a, b, c):
    """a b + c rounded to FP32 once (the FP64 product is exact)."""
    return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(np.float32)


@pytest.mark.parametrize("d,h,n", [(5, 64, 60000), (12, 48, 60000), (6, 32, 150000)])
def test_sample_sums(gpu, d, h, n):
    g = torch.Generator().manual_seed(h + d)
    half = d // 2
    W1, b1 = torch.randn(h, d, generator=g) / d ** 0.5, torch.randn(h, generator=g) * 0.1
    W2 = torch.randn(d, h, generator=g) / h ** 0.5
    zero = [torch.zeros(h, d), torch.zeros(h), torch.zeros(d, h), torch.zeros(d)]
    stats = [torch.zeros(d), torch.eye(d), torch.zeros(d), torch.eye(d)]
    theta = torch.cat([p.reshape(-1) for p in zero + [W1, b1, W2, torch.zeros(d)] + stats])
    m = RealNVP(d, 1, h, fr.PRNGKey(0), _theta=theta)
    cond, trans = list(range(half)), list(range(half, d))  # layer 0 conditions on the first half
    x = torch.randn(n, d, generator=g)
    grad, _ = m.grad_log_prob_sum(x.cuda())
    o = 2 * h * d + h + d + h * d + h  # the shift head's W2
    got = grad[o:o + d * h].cpu().reshape(d, h)[trans].numpy().astype(np.float64)

    xc, w1, w2 = x[:, cond].numpy(), W1[:, cond].numpy(), W2[trans].numpy()
    hid = np.broadcast_to(b1.numpy(), (n, h)).astype(np.float32)
    for k in range(half):
        hid = fma(xc[:, k:k + 1], w1[None, :, k], hid)
    hid = np.maximum(hid, np.float32(0))
    # y as the training pass leaves it: log N(y) has the gradient -y, read from gx of the transformed dims
    gy = m.grad_log_prob_sum(x.cuda())[1][:, trans].cpu().numpy()
    assert np.abs(gy + (x[:, trans].numpy() + hid @ w2.T)).max() < 1e-4  # (e^s = 1: gx is the gradient of y)
    exact = gy.T.astype(np.float64) @ hid.astype(np.float64)

    tiles = (n + 15) // 16
    pad = tiles * 16 - n
    a = np.pad(gy, ((0, pad), (0, 0))).reshape(tiles, 16, len(trans), 1)
    b = np.pad(hid, ((0, pad), (0, 0))).reshape(tiles, 16, 1, h)
    part = np.zeros((tiles, len(trans), h), np.float32)
    for i in range(16):
        part = fma(a[:, i], b[:, i], part)
    sums = []
    for c in range(16):
        u, mine = [np.zeros(part.shape[1:], np.float32) for _ in range(4)], part[c::16]
        for t in range(len(mine)):
            u[t % 4] = u[t % 4] + mine[t]
        sums.append((u[0] + u[1]) + (u[2] + u[3]))
    want = np.zeros_like(sums[0])
    for v in sums:
        want = want + v

    def rms(v):
        return float(np.sqrt(np.mean((v - exact) ** 2)))

    assert rms(got) <= 1.25 * rms(want.astype(np.float64))
