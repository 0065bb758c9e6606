"""gradients_fixed_kernel (values and gradients with l_max a compile-time number) against the oracle, number for number."""

import numpy as np
import pytest
import torch

from gpu_utils import announce, plan_text, run_launch_layer
from helpers import special_points
from test_gpu_parity import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("normalized", [True, False])
@pytest.mark.parametrize("l_max", range(7, 31))
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_every_l_max(oracle, library, switches, dtype, l_max, normalized):
    """The smallest and largest tile, tiles that are no power of two, one point less and more than a tile, both numbers of
    waves; arrays that start at a multiple of 16 bytes and one element past it, nothing written outside them."""
    if dtype == np.float64 and l_max > 24:
        pytest.skip("no kernel")
    ny = (l_max + 1) ** 2
    most = min(32, 160 * 1024 // (4 * (ny + 2) * np.dtype(dtype).itemsize) // 4 * 4)
    for n, tile, waves in ((1, 8, 8), (33, 8, 16), (most - 1, most, 8), (most + 1, most, 16), (50, 12, 8), (263, 20, 16)):
        library.sphx_reset_switches()
        switches("SPHX_GRADIENT_LANES_FIXED", 2)
        switches("SPHX_GRADIENT_LANES_FIXED_TILE", min(tile, most))
        switches("SPHX_GRADIENT_LANES_FIXED_WAVES", waves)
        sixteen = waves == 16 and l_max <= (16 if dtype == np.float32 else 11)
        planned = plan_text(library, n, l_max, "gradients", dtype, normalized)
        name = "double" if dtype == np.float64 else "float"
        assert planned.startswith(f"gradients_fixed_kernel<{name}, {str(normalized).lower()}, {l_max}, {16 if sixteen else 8}> "
                                  f"[l_max a constant, {min(tile, most)} points"), planned
        xyz = special_points(dtype, np.random.default_rng(l_max), n)
        want = oracle.compute(xyz, l_max, normalized, "gradients")
        for offset in (0, 1):
            announce("gradients, l_max a constant", np.dtype(dtype).name, l_max, normalized, n, tile, waves, offset)
            d_xyz = torch.from_numpy(xyz).cuda()
            out = [torch.full((n * c * ny + 2,), -7.0, dtype=d_xyz.dtype, device="cuda") for c in (1, 3)]
            views = tuple(o[offset:offset + n * c * ny] for o, c in zip(out, (1, 3))) + (None,)
            status, _ = run_launch_layer(library, d_xyz, l_max, normalized, "gradients", out=views)
            torch.cuda.synchronize()
            assert status == 0, library.sphx_last_error()
            got = tuple(v.reshape(w.shape).cpu().numpy() for v, w in zip(views[:2], want)) + (None,)
            check(got, want, (l_max, n, tile, waves, offset))
            for o in out:
                assert (o[:offset] == -7.0).all() and (o[offset - 2:] == -7.0).all()


@pytest.mark.parametrize("dtype, l_max, n", [(np.float32, 7, 9_000), (np.float32, 10, 17_001), (np.float32, 13, 131_072),
                                             (np.float32, 17, 65_536), (np.float64, 8, 10_000), (np.float64, 8, 65_537),
                                             (np.float64, 12, 65_536), (np.float64, 15, 16_384), (np.float32, 19, 65_536),
                                             (np.float32, 22, 16_384), (np.float32, 24, 4_097), (np.float64, 16, 4_097),
                                             (np.float64, 18, 5_000), (np.float64, 20, 2_049), (np.float32, 30, 2_049), (np.float64, 24, 2_049)])
def test_as_planned(oracle, library, dtype, l_max, n):
    """Calls of sizes between the table's lines, as they are planned."""
    for normalized in (True, False):
        for points in (n - 1, n):
            announce("gradients as planned", np.dtype(dtype).name, l_max, normalized, points)
            xyz = special_points(dtype, np.random.default_rng(l_max), points)
            want = oracle.compute(xyz, l_max, normalized, "gradients")
            status, out = run_launch_layer(library, torch.from_numpy(xyz).cuda(), l_max, normalized, "gradients")
            assert status == 0, library.sphx_last_error()
            check(tuple(o.cpu().numpy() if o is not None else None for o in out), want, (l_max, points))


@pytest.mark.parametrize("dtype, l_max, normalized, n, below, at", [
    # (kernel<waves> tile, or the kernel without l_max for a constant that is ahead there)
    (np.float32, 13, False, 131_072, "gradients_fixed_kernel<8> 16", "recursion_kernel"),
    (np.float32, 17, True, 65_536, "gradients_fixed_kernel<8> 12", "gradients_fixed_kernel<8> 28"),
    (np.float32, 19, True, 65_536, "gradients_fixed_kernel<8> 12", "recursion_kernel"),
    (np.float32, 22, True, 16_384, "gradients_fixed_kernel<8> 8", "recursion_kernel"),
    (np.float32, 24, False, 32_768, "gradients_fixed_kernel<8> 8", "pairs_kernel"),
    (np.float32, 30, True, 2_049, "gradients_fixed_kernel<8> 8", "recursion_kernel"),
    (np.float64, 14, True, 14_000, "gradients_fixed_kernel<8> 8", "recursion_kernel"),
    (np.float64, 15, True, 16_384, "gradients_fixed_kernel<8> 8", "recursion_kernel"),
    (np.float64, 16, True, 4_097, "gradients_fixed_kernel<8> 16", "recursion_kernel"),
    (np.float64, 18, True, 5_000, "gradients_fixed_kernel<8> 12", "recursion_kernel"),
    (np.float64, 20, True, 3_073, "gradients_fixed_kernel<8> 8", "recursion_kernel"),
    (np.float64, 19, False, 8_192, "gradients_fixed_kernel<8> 12", "recursion_kernel"),
    (np.float64, 20, False, 4_097, "gradients_fixed_kernel<8> 8", "recursion_kernel"),
    (np.float64, 24, False, 2_049, "gradients_fixed_kernel<8> 8", "recursion_kernel"),
    (np.float64, 8, False, 65_536, "gradients_fixed_kernel<8> 20", "gradients_fixed_kernel<16> 32"),
    (np.float64, 12, True, 65_536, "gradients_fixed_kernel<8> 12", "gradients_fixed_kernel<8> 28"),
])
def test_both_sides_of_the_tables_lines(oracle, library, dtype, l_max, normalized, n, below, at):
    for points, wanted in ((n - 1, below), (n, at)):
        announce("gradients at a line", np.dtype(dtype).name, l_max, normalized, points, wanted)
        planned = plan_text(library, points, l_max, "gradients", dtype, normalized)
        if "_fixed_kernel" in wanted:
            kernel, waves, tile = wanted.replace("<", " ").replace(">", "").split()
            assert planned.startswith(kernel + "<") and f", {l_max}, {waves}> [l_max a constant, {tile} points" in planned, planned
        else:
            assert planned.startswith(wanted + "<"), planned
        xyz = special_points(dtype, np.random.default_rng(l_max), points)
        want = oracle.compute(xyz, l_max, normalized, "gradients")
        status, out = run_launch_layer(library, torch.from_numpy(xyz).cuda(), l_max, normalized, "gradients")
        assert status == 0, library.sphx_last_error()
        check(tuple(o.cpu().numpy() if o is not None else None for o in out), want, (l_max, points))
