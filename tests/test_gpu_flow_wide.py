"""The wide flow pass (64-sample tiles, many samples) against the general pass:
both sum in one order, so the rows of a large call are those of small ones bit
for bit, except that calls of up to 64 samples a CU sum the wavefronts'
log-dets in another order (FP32 rounding of a sum of at most d terms of size <= 10:
2^-24 * 10 * d a layer). Reference: src/flowMC/resource/model/nf_model/rqSpline.py:450-504.
"""

import ctypes as C

import pytest
import torch

from flowmc_amd import _native as N
from flowmc_amd import random as fr
from flowmc_amd.resource.model.nf_model.rqSpline import MaskedCouplingRQSpline

pytestmark = pytest.mark.gpu

SMALL = 4096  # samples a call of the general pass


def _model(d, layers, hidden, bins):
    m = MaskedCouplingRQSpline(d, layers, hidden, bins, fr.PRNGKey(d + bins), precision="bfloat16")
    g = torch.Generator().manual_seed(d)
    m.theta.add_(0.05 * torch.randn(m.theta.numel(), generator=g).cuda() * (m.theta != 1))
    m._stat("data_cov").copy_(torch.diag(0.5 + torch.rand(d, generator=g)))
    m._stat("base_cov").copy_(torch.eye(d))
    m.mark_updated()
    m._ensure_packed()
    return m


def _pass(m, direction, flags, x, n, d, first=0):
    s = m._struct()
    y, ld = torch.full((n, d), float("nan"), device="cuda"), torch.full((n,), float("nan"), device="cuda")
    N.call("fmc_flow_pass", N.stream_ptr(), C.byref(s), direction, flags, None if x is None else x.data_ptr(), n, 3, 4,
           first, y.data_ptr(), ld.data_ptr(), None, None, None)
    return y, ld


# n: the first with the wide pass for broad / other conditioners on 256 CUs
# leave ragged last tiles; widths of one to four layers, odd d, blocks of
# wavefronts without a share, k-steps that are no multiple of the ring
@pytest.mark.parametrize("d,layers,hidden,bins,n", [
    (64, 2, [256, 256], 8, 16385), (2, 3, [32, 32], 8, 41001), (7, 3, [64], 10, 41024), (33, 2, [128, 256, 64, 32], 8, 40961),
    (9, 2, [96, 32, 64], 5, 41063), (3, 2, [40, 70], 3, 41000), (100, 2, [200, 256], 8, 16449), (16, 2, [160], 10, 20001),
])
# forward with standardisation and base log-prob, reference inverse from base
# draws, exact inverse with the log-density from draws and from given rows
@pytest.mark.parametrize("direction,flags,draws", [(0, 3, False), (1, 5, True), (2, 7, True), (2, 4, False)])
def test_wide_pass_rows_match_the_general_pass(gpu, direction, flags, draws, d, layers, hidden, bins, n):
    m = _model(d, layers, hidden, bins)
    x = None if draws else 3 * torch.randn(n, d, generator=torch.Generator().manual_seed(n)).cuda()
    y, ld = _pass(m, direction, flags, x, n, d)
    for a in (0, n // 2, n - SMALL):
        ys, ls = _pass(m, direction, flags, None if draws else x[a:a + SMALL].contiguous(), SMALL, d, a)
        assert torch.equal(y[a:a + SMALL], ys)
        assert ((ld[a:a + SMALL] - ls).abs() <= 2.0 ** -24 * 10 * d * (layers + 1)).all()


# n at the rounds in which 256 CUs take a call (96 samples a CU in the general
# pass, 128 in the wide one), for conditioners on either side of each rule
@pytest.mark.parametrize("n", [24576, 24577, 32768, 32769, 49153, 73729])
@pytest.mark.parametrize("d,layers,hidden,bins", [
    (2, 2, [32, 32], 8), (33, 2, [128, 256, 64, 32], 8), (7, 2, [64], 10), (16, 2, [100, 70], 5), (8, 2, [256], 8),
])
@pytest.mark.parametrize("direction,flags,draws", [(0, 3, False), (2, 7, True)])
def test_rows_around_the_rounds_match_small_calls(gpu, direction, flags, draws, d, layers, hidden, bins, n):
    m = _model(d, layers, hidden, bins)
    x = None if draws else 3 * torch.randn(n, d, generator=torch.Generator().manual_seed(n)).cuda()
    y, ld = _pass(m, direction, flags, x, n, d)
    for a in (0, n // 2, n - SMALL):
        ys, ls = _pass(m, direction, flags, None if draws else x[a:a + SMALL].contiguous(), SMALL, d, a)
        assert torch.equal(y[a:a + SMALL], ys)
        assert ((ld[a:a + SMALL] - ls).abs() <= 2.0 ** -24 * 10 * d * (layers + 1)).all()
