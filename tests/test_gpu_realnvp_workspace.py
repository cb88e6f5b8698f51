"""The workspace of the RealNVP backward sweep is bounded, and a sweep that takes
few layers at a time, or several tiles a workgroup, has the gradients of the
per-layer calls (the same FP32 terms in another order: 1e-5 of the largest entry
covers 2^-24 sqrt(n) of sums of 10^4 samples; 3e-5 for 10^5). Reference:
src/flowMC/resource/model/nf_model/base.py:98-125.
"""

import ctypes as C

import pytest
import torch

from flowmc_amd import _native as N
from flowmc_amd import random as fr
from flowmc_amd.resource.model.nf_model.realNVP import RealNVP

pytestmark = pytest.mark.gpu


# a launch a layer; all layers in one; several tiles a workgroup: ragged
# counts of tiles of one and of three groups of 16 samples
@pytest.mark.parametrize("d,L,h,n,tol", [(128, 4, 250, 8200, 1e-5), (130, 3, 20, 9001, 1e-5), (5, 2, 20, 60001, 3e-5),
                                         (20, 2, 33, 30007, 3e-5)])
def test_sweep_in_parts(gpu, d, L, h, n, tol):
    m = RealNVP(d, L, h, fr.PRNGKey(d))
    m.theta.add_(0.05 * torch.randn(m.theta.numel(), generator=torch.Generator().manual_seed(d)).cuda() * (m.theta.abs() < 0.9))
    m.mark_updated()
    m._ensure_packed()
    x = torch.randn(n, d, generator=torch.Generator().manual_seed(n)).cuda()
    got, ggx = m.grad_log_prob_sum(x)

    s = m._struct()
    per, tile = C.c_int64(), C.c_int32()
    N.call("fmc_rnvp_sizes", C.byref(s), None, None, C.byref(per), C.byref(tile))
    tiles = (n + tile.value - 1) // tile.value
    one = torch.ones(n, device="cuda")
    saved, gy, gx = torch.empty(L, n, d, device="cuda"), torch.empty(n, d, device="cuda"), torch.empty(n, d, device="cuda")
    N.call("fmc_rnvp_pass", N.stream_ptr(), C.byref(s), 0, 3, x.data_ptr(), n, 0, 0, 0, None, None, saved.data_ptr(),
           one.data_ptr(), gy.data_ptr())
    part, want = torch.empty((tiles + 16) * per.value, device="cuda"), torch.zeros_like(m.theta)
    for layer in reversed(range(L)):
        N.call("fmc_rnvp_backward_layer", N.stream_ptr(), C.byref(s), layer, saved[layer].data_ptr(), n, one.data_ptr(),
               gy.data_ptr(), gx.data_ptr(), part.data_ptr(), tiles)
        N.call("fmc_rnvp_weight_grad", N.stream_ptr(), C.byref(s), layer, part.data_ptr(), tiles, tiles + 16,
               want.data_ptr())
        gy, gx = gx, gy
    assert float((got - want).abs().max()) <= tol * float(want.abs().max())
    gy = gy / torch.sqrt(torch.diagonal(m.data_cov))
    assert float((ggx - gy).abs().max()) <= 1e-5 * float(gy.abs().max())
