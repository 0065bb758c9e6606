"""values_kernel with eight channels side by side in a wave (tiles of eight points), and the shapes the planner gives
that form, four channels or two, against the oracle, number for number: the same operations in the same order."""

import numpy as np
import pytest
import torch

from gpu_utils import announce, run_launch_layer
from helpers import special_points
from test_gpu_parity import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("l_max", [7, 8, 13, 14, 15, 16, 18, 23, 24, 26, 28, 32, 34, 41])
@pytest.mark.parametrize("pack", [8, None])
def test_bundles_of_channels(oracle, library, switches, dtype, l_max, pack):
    """Channels that leave the last bundle partly empty (l_max = 7: seven of eight), one step above the closed forms,
    padded rows (l_max = 15, 23), tiles with one point, one short of full, full, and one more."""
    rng = np.random.default_rng(61)
    library.sphx_reset_switches()
    switches("SPHX_VALUES_FIXED", 0)  # (not the kernels with l_max for a constant)
    if pack is not None:
        switches("SPHX_VALUES_PACK", pack)
        switches("SPHX_PAIRS", 0)
    for normalized in (True, False):
        for n in (1, 7, 8, 9, 1201):
            xyz = special_points(dtype, rng, n)
            want = oracle.compute(xyz, l_max, normalized, "values")
            announce("values, bundles", np.dtype(dtype).name, normalized, l_max, n, "pack", pack)
            status, got = run_launch_layer(library, torch.from_numpy(xyz).cuda(), l_max, normalized, "values")
            torch.cuda.synchronize()
            assert status == 0, library.sphx_last_error()
            check(tuple(None if g is None else g.cpu().numpy() for g in got), want, (l_max, normalized, n, pack))
    library.sphx_reset_switches()
