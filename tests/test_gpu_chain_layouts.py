"""The chain kernels that the launch rules choose between, against each other:
random numbers drawn by the chain's own wavefront, by other wavefronts of the
workgroup (few chains), or injected; lane counts compiled in or taken at run
time (workgroups above 256 threads). All of them round alike, so that outputs
are compared bit for bit. Reference: src/flowMC/resource/kernel/MALA.py:26-89,
Gaussian_random_walk.py:25-61, strategy/parallel_tempering.py:291-372.
"""

import ctypes as C

import pytest
import torch

from flowmc_amd import _native as N
from flowmc_amd import targets as TG
from oracle import philox as OP
from oracle import tempering as OPT

pytestmark = pytest.mark.gpu

KEY = (0x1234, 0x9876)


def _target(name, d):
    g = torch.Generator().manual_seed(d)
    kind, _, k = name.partition(":")
    if kind == "dense":
        a = torch.randn(d, d, generator=g, dtype=torch.float64)
        return TG.GaussianDense(torch.randn(d, generator=g, dtype=torch.float64), a @ a.T / d + torch.eye(d))
    if kind == "gmm":
        means = 3 * torch.randn(int(k), d, generator=g, dtype=torch.float64)
        return TG.GaussianMixtureDiag(means, 0.5 + torch.rand(int(k), d, generator=g, dtype=torch.float64))
    return {"diag": lambda: TG.GaussianDiag(torch.zeros(d), torch.ones(d)), "rosenbrock": lambda: TG.Rosenbrock(d),
            "funnel": lambda: TG.Funnel(d)}[kind]()


def _run(entry, t, x0, steps, step0, thinning, noise=None, log_u=None, block=0):
    n, d = x0.shape
    rows = (step0 + steps - 1) // thinning + 1
    x, lp = x0.clone(), torch.zeros(n, device="cuda")
    outs = [torch.zeros(n, rows, d, device="cuda"), torch.zeros(n, rows, device="cuda"),
            torch.zeros(n, rows, device="cuda")]
    cfg = C.byref(N.fmc_launch_cfg(0, 0, block, 0)) if block else None
    ptr = [None if z is None else z.data_ptr() for z in (noise, log_u)]
    desc = t.descriptor()
    N.call(entry, N.stream_ptr(), C.byref(desc), x.data_ptr(), lp.data_ptr(), n, steps, step0, 0.03, *KEY, *ptr,
           *(o.data_ptr() for o in outs), rows, 0, thinning, cfg)
    return [x, lp] + outs


# d = 128 Rosenbrock: 4 chains a wavefront, so 4096 chains are the last that
# have their random numbers drawn by other wavefronts. 64-D mixtures: the
# parameters of 62 modes leave just room for those in LDS, of 63 none.
@pytest.mark.parametrize("name,d,n,steps,step0,thinning", [
    ("dense", 1, 1, 15, 0, 1), ("dense", 4, 65, 16, 3, 1), ("dense", 5, 63, 8, 0, 1), ("dense", 5, 64, 9, 2, 3),
    ("dense", 7, 1000, 7, 0, 1), ("dense", 12, 130, 13, 0, 1), ("dense", 33, 20, 17, 0, 1),
    ("diag", 3, 129, 33, 0, 2), ("diag", 6, 33, 17, 1, 1), ("diag", 256, 3, 31, 0, 1),
    ("rosenbrock", 2, 64, 16, 0, 1), ("rosenbrock", 31, 17, 17, 0, 1), ("rosenbrock", 128, 4096, 9, 0, 4),
    ("rosenbrock", 128, 4097, 9, 0, 4), ("rosenbrock", 512, 2, 24, 0, 1), ("funnel", 7, 301, 18, 0, 1),
    ("funnel", 130, 5, 32, 0, 1), ("gmm:1", 1, 70, 16, 0, 1), ("gmm:3", 17, 50, 19, 0, 1), ("gmm:62", 64, 9, 20, 0, 1),
    ("gmm:63", 64, 9, 20, 0, 1),
])
@pytest.mark.parametrize("entry,sid_n,sid_u", [("fmc_mala_run", OP.RNG_MALA_NOISE, OP.RNG_MALA_UNIFORM),
                                               ("fmc_grw_run", OP.RNG_GRW_NOISE, OP.RNG_GRW_UNIFORM)])
def test_chain_kernels_agree(gpu, entry, sid_n, sid_u, name, d, n, steps, step0, thinning):
    t = _target(name, d)
    x0 = torch.randn(n, d, generator=torch.Generator().manual_seed(n)).cuda() * 0.5
    noise, lu = torch.empty(steps, n, d, device="cuda"), torch.empty(steps, n, device="cuda")
    N.call("fmc_rng_normal", N.stream_ptr(), *KEY, n, d, steps, step0, sid_n, noise.data_ptr())
    N.call("fmc_rng_log_uniform", N.stream_ptr(), *KEY, n, steps, step0, sid_u, lu.data_ptr())
    want = _run(entry, t, x0, steps, step0, thinning, noise, lu)
    assert all(torch.isfinite(w).all() for w in want)
    for block in (0, 64, 512):  # launch rules' own choice; own draws; lane count at run time
        got = _run(entry, t, x0, steps, step0, thinning, block=block)
        for a, b in zip(want, got):
            assert torch.equal(a, b), f"block {block}"


@pytest.mark.parametrize("n,T,d,off", [(7, 3, 4, 0), (8, 2, 8, 0), (9, 5, 12, 0), (17, 4, 8, 1), (8, 64, 4, 3)])
def test_exchange_rows_at_block_edges(gpu, n, T, d, off):
    """Rows move bit for bit; rows that start off a 16-byte boundary too."""
    g = torch.Generator().manual_seed(n * T)
    x = torch.randn(n, T, d, generator=g)
    L = (torch.randn(n, T, generator=g) * 3).float()
    lu = torch.log(torch.rand(n, T - 1, generator=g))
    temps = torch.linspace(1.0, 6.0, T)
    buf, out = (torch.full((n * T * d + off,), float("nan"), device="cuda") for _ in range(2))
    buf[off:] = x.reshape(-1).cuda()
    Lg, acc, tg, lg = L.cuda(), torch.empty(n, T - 1, device="cuda"), temps.cuda(), lu.cuda()
    N.call("fmc_pt_exchange", N.stream_ptr(), buf[off:].data_ptr(), out[off:].data_ptr(), Lg.data_ptr(),
           tg.data_ptr(), n, T, d, 0, 0, lg.data_ptr(), acc.data_ptr())
    y, Ly, ra = OPT.exchange(x.double(), L.double(), temps.double(), lu.double())
    ok = (acc.cpu().bool() == ra).all(1)  # (a decision within rounding of its log u may differ)
    assert int((~ok).sum()) <= 1
    assert torch.equal(out[off:].cpu().reshape(n, T, d)[ok], y[ok].float())
    assert torch.equal(Lg.cpu()[ok], Ly[ok].float())
