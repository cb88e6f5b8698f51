"""Every form of the chain kernels for long vectors and explicit layouts (rows or
the unpadded block in LDS or memory, workgroups of at most 256 threads or more,
few and many workgroups): the log-density a chain ends on is the FP64 oracle's at
the position it ends on (FP32 sums of d terms: 2e-5 relative), and chains of a
call do not depend on how many there are beside them.
Reference: src/flowMC/resource/kernel/MALA.py:26-89, HMC.py:41-118.
"""

import ctypes as C

import pytest
import torch

from flowmc_amd import _native as N
from flowmc_amd import targets as TG
from oracle import targets as OT

pytestmark = pytest.mark.gpu


def _target(name, d):
    g = torch.Generator().manual_seed(d)
    mean = torch.randn(d, generator=g, dtype=torch.float64).float().double()
    if name == "gmm":
        means = torch.randn(8, d, generator=g, dtype=torch.float64).float().double()
        sig = torch.ones(8, d, dtype=torch.float64)
        return TG.GaussianMixtureDiag(means, sig), lambda x: OT.gmm_diag(x, means, sig)
    if name == "diag":
        return TG.GaussianDiag(mean, torch.ones(d)), lambda x: OT.gauss_diag(x, mean, torch.ones(d, dtype=torch.float64))
    if name == "dense":
        p = torch.eye(d, dtype=torch.float64) + 0.5 / d
        p = p.float().double()
        return TG.GaussianDense(mean, p), lambda x: OT.gauss_dense(x, mean, p)
    return (TG.Rosenbrock(d), OT.rosenbrock) if name == "ros" else (TG.Funnel(d), OT.funnel)


@pytest.mark.parametrize("name,d,n,cfg", [
    ("gmm", 300, 100, None), ("gmm", 300, 10000, None), ("gmm", 300, 41, (0, 0, 512, 0)), ("gmm", 600, 41, None),
    ("gmm", 600, 41, (0, 0, 512, 0)), ("gmm", 64, 41, (64, 1, 256, 0)), ("gmm", 64, 300, (64, 1, 256, 0)),
    ("gmm", 20, 100, (8, 2, 512, 0)), ("diag", 600, 41, None), ("diag", 600, 41, (0, 0, 512, 0)), ("diag", 1500, 41, None),
    ("diag", 1500, 41, (0, 0, 512, 0)), ("diag", 30, 41, (1, 8, 64, 0)), ("diag", 100, 41, (64, 1, 256, 0)),
    ("ros", 700, 41, None), ("ros", 1500, 41, (0, 0, 512, 0)), ("fun", 600, 41, None), ("fun", 1500, 41, (0, 0, 512, 0)),
    ("dense", 130, 41, None), ("dense", 60, 41, (16, 8, 256, 0)),
])
def test_chains_end_on_the_log_density_of_their_position(gpu, name, d, n, cfg):
    t, fn = _target(name, d)
    desc, few = t.descriptor(), 40
    x0 = (0.3 * torch.randn(n, d, generator=torch.Generator().manual_seed(n))).cuda()
    cf = None if cfg is None else C.byref(N.fmc_launch_cfg(*cfg))

    def run(entry, m):
        x, lp, acc = x0[:m].clone(), torch.empty(m, device="cuda"), torch.zeros(m, 12, device="cuda")
        step = (12, 0, 1e-3) if entry != "fmc_hmc_run" else (12, 0, 1e-3, 5, None, None)
        N.call(entry, N.stream_ptr(), C.byref(desc), x.data_ptr(), lp.data_ptr(), m, *step, 1, 2, None, None, None, None,
               acc.data_ptr(), 12, 0, 1, cf)
        return x, lp, acc

    for entry in ("fmc_mala_run", "fmc_grw_run", "fmc_hmc_run"):
        x, lp, acc = run(entry, n)
        assert float(acc.mean()) > 0.5
        rows = torch.cat([torch.arange(few), torch.arange(n - few, n)])
        v = fn(x.cpu().double()[rows])
        assert ((lp.cpu().double()[rows] - v).abs() <= 2e-5 * (1 + v.abs())).all()
        xs, ls, accs = run(entry, few)
        same = (accs == acc[:few]).all(1)  # (another form rounds otherwise: a decision may fall differently)
        assert int(same.sum()) >= few - 2
        assert torch.allclose(xs[same], x[:few][same], rtol=1e-4, atol=1e-4)
