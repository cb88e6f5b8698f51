"""Rosenbrock's value and gradient for every lane count and for dims whose last
chunk, lane or half of a wavefront is ragged, against the FP64 oracle: each
element reads its neighbours across chunks and lanes. FP32 sums of d terms: 2e-5
relative. Reference: the jax.grad of the target at src/flowMC/resource/kernel/MALA.py:59.
"""

import ctypes as C

import pytest
import torch

from flowmc_amd import _native as N
from flowmc_amd import targets as TG
from oracle import targets as OT

pytestmark = pytest.mark.gpu

LAYOUTS = [None] + [(lanes, chunks) for lanes in (1, 2, 4, 8, 16, 32, 64) for chunks in (1, 2, 4)]


@pytest.mark.parametrize("d", [2, 5, 8, 13, 31, 33, 64, 95, 127, 200, 250, 511, 512])
def test_value_and_gradient(gpu, d):
    t = TG.Rosenbrock(d)
    x = (1.0 + 0.4 * torch.randn(37, d, generator=torch.Generator().manual_seed(d), dtype=torch.float64)).float()
    v, g = OT.value_and_grad(OT.rosenbrock, x.double())
    xg, desc, ran = x.cuda(), t.descriptor(), 0
    for layout in LAYOUTS:
        if layout is not None and not d <= 4 * layout[0] * layout[1] < 32 * d:
            continue
        cfg = None if layout is None else C.byref(N.fmc_launch_cfg(*layout, 256, 0))
        lp, gr = torch.empty(37, device="cuda"), torch.full((37, d), float("nan"), device="cuda")
        N.call("fmc_target_eval", N.stream_ptr(), C.byref(desc), xg.data_ptr(), 37, lp.data_ptr(), gr.data_ptr(), cfg)
        assert ((lp.cpu().double() - v).abs() <= 2e-5 * (1 + v.abs())).all(), layout
        assert ((gr.cpu().double() - g).abs() <= 2e-5 * (1 + g.abs().amax(-1, keepdim=True))).all(), layout
        # the fused steps' evaluation at their entry and at a rejected proposal's end is the same value
        y, end, acc = xg.clone(), torch.empty(37, device="cuda"), torch.zeros(37, 8, device="cuda")
        N.call("fmc_mala_run", N.stream_ptr(), C.byref(desc), y.data_ptr(), end.data_ptr(), 37, 8, 0, 0.01, 1, 2, None, None,
               None, None, acc.data_ptr(), 8, 0, 1, cfg)
        ve = OT.rosenbrock(y.cpu().double())
        assert int(acc.sum()) > 37 and ((end.cpu().double() - ve).abs() <= 2e-5 * (1 + ve.abs())).all(), layout
        ran += 1
    assert ran >= 3
