"""RealNVP library calls that end on the host (no GPU needed)."""

import ctypes as C

import pytest

from flowmc_amd import _native as N

FAKE = 0x1000  # never read: the calls are refused before a launch


def _flow(d, L, h):
    return N.fmc_rnvp(d, L, h, 1.0, FAKE, FAKE, FAKE)


@pytest.mark.parametrize("tiles", [1, 16, 17, 255, 256, 4096])
def test_weight_grad_refuses_too_few_rows(tiles):
    rows = tiles + min(16, (tiles + 15) // 16)
    with pytest.raises(N.FlowMCNativeError, match="partials hold"):
        N.call("fmc_rnvp_weight_grad", None, C.byref(_flow(5, 2, 20)), 0, FAKE, tiles, rows - 1, FAKE)
