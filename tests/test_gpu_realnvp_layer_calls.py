"""The per-layer adjoint calls of the library (fmc_rnvp_backward_layer,
fmc_rnvp_weight_grad) against the one-call sweep (fmc_rnvp_backward): the same
FP32 terms added in another order, so that a sum of n samples differs by a few
2^-24 sqrt(n) of its largest terms; 1e-5 of the largest entry covers n <= 10^4.
Reference: src/flowMC/resource/model/nf_model/base.py:98-125.
"""

import ctypes as C

import pytest
import torch

from flowmc_amd import _native as N
from flowmc_amd import random as fr
from flowmc_amd.resource.model.nf_model.realNVP import RealNVP

pytestmark = pytest.mark.gpu


def _forward(m, x, g_logp):
    d, L, n = m.n_features, m.n_layers, x.shape[0]
    saved, gy = torch.empty(L, n, d, device="cuda"), torch.empty(n, d, device="cuda")
    N.call("fmc_rnvp_pass", N.stream_ptr(), C.byref(m._struct()), 0, 3, x.data_ptr(), n, 0, 0, 0, None, None,
           saved.data_ptr(), g_logp.data_ptr(), gy.data_ptr())
    return saved, gy


# one, two and three groups of 16 samples a tile in the sweep; batches in one
# to three calls whose rows follow one another; partials off a 16-byte boundary
@pytest.mark.parametrize("d,L,h,parts,off", [(5, 2, 20, [40], 0), (5, 2, 20, [3000, 2500], 1), (33, 3, 40, [4500, 17, 5000], 0),
                                             (40, 2, 100, [8200], 3), (70, 2, 20, [33, 100], 2)])
def test_layer_calls_sum_to_the_sweep(gpu, d, L, h, parts, off):
    m = RealNVP(d, L, h, fr.PRNGKey(d))
    m.theta.add_(0.1 * torch.randn(m.theta.numel(), generator=torch.Generator().manual_seed(d)).cuda() * (m.theta.abs() < 0.9))
    m.mark_updated()
    m._ensure_packed()
    n = sum(parts)
    g = torch.Generator().manual_seed(n)
    x, w = torch.randn(n, d, generator=g).cuda(), (torch.rand(n, generator=g) + 0.5).cuda()
    want, _ = m.grad_log_prob_sum(x, w)

    s = m._struct()
    per, tile = C.c_int64(), C.c_int32()
    N.call("fmc_rnvp_sizes", C.byref(s), None, None, C.byref(per), C.byref(tile))
    tiles = [(k + tile.value - 1) // tile.value for k in parts]
    rows = sum(tiles) + min(16, (sum(tiles) + 15) // 16)
    grad, gxs = torch.zeros_like(m.theta), []
    state = []
    for a, k in zip([sum(parts[:i]) for i in range(len(parts))], parts):
        xa, wa = x[a:a + k].contiguous(), w[a:a + k].contiguous()
        state.append([wa, *_forward(m, xa, wa), torch.empty(k, d, device="cuda")])
    for layer in reversed(range(L)):
        part = torch.full((rows * per.value + off,), float("nan"), device="cuda")
        at = 0
        for st, t in zip(state, tiles):
            wa, saved, gy, gx = st
            k = gy.shape[0]
            N.call("fmc_rnvp_backward_layer", N.stream_ptr(), C.byref(s), layer, saved[layer].data_ptr(), k, wa.data_ptr(),
                   gy.data_ptr(), gx.data_ptr(), part.data_ptr() + 4 * (off + at * per.value), t)
            st[2], st[3] = gx, gy
            at += t
        N.call("fmc_rnvp_weight_grad", N.stream_ptr(), C.byref(s), layer, part.data_ptr() + 4 * off, at, rows,
               grad.data_ptr())
    assert float((grad - want).abs().max()) <= 1e-5 * float(want.abs().max())
