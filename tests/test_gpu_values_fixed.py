"""values_fixed_kernel (values with l_max a compile-time number) against the oracle, number for number."""

import numpy as np
import pytest
import torch

from gpu_utils import announce, plan_text, run_launch_layer
from helpers import special_points
from test_gpu_parity import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("normalized", [True, False])
@pytest.mark.parametrize("l_max", range(7, 33))
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_every_l_max(oracle, library, switches, dtype, l_max, normalized):
    """The smallest and largest tile, tiles that are no power of two, one point less and more than a tile, both numbers of
    waves; arrays that start at a multiple of 16 bytes and one element past it, nothing written outside them."""
    if dtype == np.float64 and l_max > 28:
        pytest.skip("no kernel")
    ny = (l_max + 1) ** 2
    most = min(32, 160 * 1024 // ((ny + 2) * np.dtype(dtype).itemsize) // 4 * 4)
    for n, tile, waves in ((1, 4, 8), (33, 8, 4), (most - 1, most, 8), (most + 1, most, 4), (50, 12, 8), (263, 20, 4)):
        library.sphx_reset_switches()
        switches("SPHX_VALUES_FIXED", 2)
        switches("SPHX_VALUES_FIXED_TILE", min(tile, most))
        switches("SPHX_VALUES_FIXED_WAVES", waves)
        planned = plan_text(library, n, l_max, "values", dtype, normalized)
        name = "double" if dtype == np.float64 else "float"
        assert planned.startswith(f"values_fixed_kernel<{name}, {str(normalized).lower()}, {l_max}, {waves}> "
                                  f"[l_max a constant, {min(tile, most)} points"), planned
        xyz = special_points(dtype, np.random.default_rng(l_max), n)
        want = oracle.compute(xyz, l_max, normalized, "values")
        for offset in (0, 1):
            announce("values, l_max a constant", np.dtype(dtype).name, l_max, normalized, n, tile, waves, offset)
            d_xyz = torch.from_numpy(xyz).cuda()
            out = torch.full((n * ny + 2,), -7.0, dtype=d_xyz.dtype, device="cuda")
            view = out[offset:offset + n * ny]
            status, _ = run_launch_layer(library, d_xyz, l_max, normalized, "values", out=(view, None, None))
            torch.cuda.synchronize()
            assert status == 0, library.sphx_last_error()
            check((view.reshape(want[0].shape).cpu().numpy(), None, None), want, (l_max, n, tile, waves, offset))
            assert (out[:offset] == -7.0).all() and (out[offset - 2:] == -7.0).all()


@pytest.mark.parametrize("dtype, l_max, n", [(np.float32, 7, 9_000), (np.float32, 12, 32_768), (np.float32, 26, 6_144),
                                             (np.float32, 26, 32_768), (np.float32, 21, 16_385), (np.float32, 32, 16_384),
                                             (np.float64, 9, 65_537), (np.float64, 18, 6_144), (np.float64, 22, 32_768),
                                             (np.float64, 25, 20_000), (np.float64, 28, 4_097), (np.float64, 29, 3_000)])
def test_as_planned(oracle, library, dtype, l_max, n):
    """Calls of sizes between the table's lines, as they are planned."""
    for normalized in (True, False):
        for points in (n - 1, n):
            announce("values as planned", np.dtype(dtype).name, l_max, normalized, points)
            xyz = special_points(dtype, np.random.default_rng(l_max), points)
            want = oracle.compute(xyz, l_max, normalized, "values")
            status, out = run_launch_layer(library, torch.from_numpy(xyz).cuda(), l_max, normalized, "values")
            assert status == 0, library.sphx_last_error()
            check(tuple(o.cpu().numpy() if o is not None else None for o in out), want, (l_max, points))


@pytest.mark.parametrize("dtype, l_max, normalized, n, below, at", [
    # (kernel<waves> tile, or the kernel without l_max for a constant that is ahead there)
    (np.float32, 24, False, 65_536, "values_fixed_kernel<8> 16", "values_fixed_kernel<8> 24"),
    (np.float32, 18, True, 262_144, "values_fixed_kernel<8> 20", "values_kernel"),
    (np.float32, 10, False, 524_288, "values_fixed_kernel<8> 32", "values_kernel"),
    (np.float64, 12, True, 300_000, "values_fixed_kernel<8> 32", "values_kernel"),
    (np.float32, 13, False, 400_000, "values_fixed_kernel<8> 24", "values_kernel"),
])
def test_both_sides_of_the_tables_lines(oracle, library, dtype, l_max, normalized, n, below, at):
    for points, wanted in ((n - 1, below), (n, at)):
        announce("values at a line", np.dtype(dtype).name, l_max, normalized, points, wanted)
        planned = plan_text(library, points, l_max, "values", dtype, normalized)
        if "_fixed_kernel" in wanted:
            kernel, waves, tile = wanted.replace("<", " ").replace(">", "").split()
            assert planned.startswith(kernel + "<") and f", {l_max}, {waves}> [l_max a constant, {tile} points" in planned, planned
        else:
            assert planned.startswith(wanted + "<"), planned
        xyz = special_points(dtype, np.random.default_rng(l_max), points)
        want = oracle.compute(xyz, l_max, normalized, "values")
        status, out = run_launch_layer(library, torch.from_numpy(xyz).cuda(), l_max, normalized, "values")
        assert status == 0, library.sphx_last_error()
        check(tuple(o.cpu().numpy() if o is not None else None for o in out), want, (l_max, points))
