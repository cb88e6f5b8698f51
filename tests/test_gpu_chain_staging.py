"""Targets whose parameters fit the LDS only as they are (rows padded to the
lanes' dims would exceed 64 KB): value and gradient against the FP64 oracle, and
fused steps that end on the log-density of their last position bit for bit (every
evaluation at a proposal rounds alike). Tolerances: FP32 sums of d terms, 2e-5
relative; the mixture's mode weights move by u |q| ~ 1e-5 relative and its
gradient by that times the spread of the modes' gradients (~10), 1e-4.
Reference: src/flowMC/resource/kernel/MALA.py:26-89.
"""

import ctypes as C

import pytest
import torch

from flowmc_amd import _native as N
from flowmc_amd import targets as TG
from oracle import targets as OT

pytestmark = pytest.mark.gpu


def _target(name, d, k):
    g = torch.Generator().manual_seed(d + k)
    if name == "dense":
        a = torch.randn(d, d, generator=g, dtype=torch.float64)
        mean, p = torch.randn(d, generator=g, dtype=torch.float64), a @ a.T / d + torch.eye(d, dtype=torch.float64)
        mean, p = mean.float().double(), p.float().double()
        return TG.GaussianDense(mean, p), lambda x: OT.gauss_dense(x, mean, p), mean
    means = torch.randn(k, d, generator=g, dtype=torch.float64)
    sig = 0.5 + torch.rand(k, d, generator=g, dtype=torch.float64)
    t = TG.GaussianMixtureDiag(means, sig)
    return t, lambda x: OT.gmm_diag(x, means, sig), means[0]


# the sizes around the limit: rows fit / the block alone / neither
@pytest.mark.parametrize("name,d,k", [("gmm", 65, 63), ("gmm", 65, 64), ("gmm", 65, 93), ("gmm", 65, 94), ("gmm", 33, 150),
                                      ("gmm", 3, 1500), ("dense", 96, 0), ("dense", 110, 0), ("dense", 127, 0), ("dense", 128, 0)])
def test_parameters_that_fit_unpadded(gpu, name, d, k):
    t, fn, start = _target(name, d, k)
    x64 = start + torch.randn(130, d, generator=torch.Generator().manual_seed(1), dtype=torch.float64)
    x = x64.float().cuda()
    lp, gr = torch.empty(130, device="cuda"), torch.empty_like(x)
    desc = t.descriptor()
    N.call("fmc_target_eval", N.stream_ptr(), C.byref(desc), x.data_ptr(), 130, lp.data_ptr(), gr.data_ptr(), None)
    v, g = OT.value_and_grad(fn, x.cpu().double())
    assert ((lp.cpu().double() - v).abs() <= 2e-5 * (1 + v.abs())).all()
    tol = 1e-4 if name == "gmm" else 2e-5
    assert ((gr.cpu().double() - g).abs() <= tol * (1 + g.abs().amax(-1, keepdim=True))).all()
    for entry in ("fmc_mala_run", "fmc_grw_run"):
        y, end = x.clone(), torch.empty(130, device="cuda")
        acc = torch.zeros(130, 12, device="cuda")
        N.call(entry, N.stream_ptr(), C.byref(desc), y.data_ptr(), end.data_ptr(), 130, 12, 0, 0.05, 1, 2, None, None, None,
               None, acc.data_ptr(), 12, 0, 1, None)
        N.call("fmc_target_eval", N.stream_ptr(), C.byref(desc), y.data_ptr(), 130, lp.data_ptr(), None, None)
        moved = acc.any(1)
        assert int(moved.sum()) > 65
        assert torch.equal(end[moved], lp[moved])


@pytest.mark.parametrize("d", [1, 2, 3, 4, 5, 7, 9, 18, 33, 110])
def test_dense_gaussian_at_infinity(gpu, d):
    """Every entry of the precision and of x - mean positive: the log-density is
    -inf, and so is every entry of the gradient."""
    p = torch.eye(d, dtype=torch.float64) + 0.5
    t = TG.GaussianDense(torch.zeros(d, dtype=torch.float64), p)
    x = torch.ones(d, d) + torch.diag(torch.full((d,), float("inf")))
    lp, gr = torch.empty(d, device="cuda"), torch.empty(d, d, device="cuda")
    desc, xg = t.descriptor(), x.cuda()
    N.call("fmc_target_eval", N.stream_ptr(), C.byref(desc), xg.data_ptr(), d, lp.data_ptr(), gr.data_ptr(), None)
    assert torch.equal(lp.cpu(), torch.full((d,), -float("inf")))
    assert torch.equal(gr.cpu(), torch.full((d, d), -float("inf")))
    for cfg in (None, N.fmc_launch_cfg(1, 2, 256, 0)):  # two chunks a lane: also with padding in both
        if cfg is not None and d > 8:
            continue
        y, end = xg.clone(), torch.empty(d, device="cuda")  # a chain that starts there keeps its state
        N.call("fmc_mala_run", N.stream_ptr(), C.byref(desc), y.data_ptr(), end.data_ptr(), d, 3, 0, 0.05, 1, 2, None, None,
               None, None, None, 0, 0, 1, None if cfg is None else C.byref(cfg))
        assert torch.equal(y, xg) and torch.equal(end.cpu(), lp.cpu())
