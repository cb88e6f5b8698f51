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


@pytest.mark.parametrize("d,L,h", [(5, 4, 64), (32, 8, 256), (64, 10, 256), (128, 10, 256), (200, 6, 500)])
@pytest.mark.parametrize("n", [1, 10000, 409600, 10 ** 8])
def test_backward_workspace_is_bounded(d, L, h, n):
    """256 MB, or one layer's gradients for two workgroups a CU."""
    size, per = C.c_int64(), C.c_int64()
    N.call("fmc_rnvp_backward_ws_size", C.byref(_flow(d, L, h)), n, C.byref(size))
    N.call("fmc_rnvp_sizes", C.byref(_flow(d, L, h)), None, None, C.byref(per), None)
    assert size.value <= max(64 << 20, 512 * per.value)
