"""hessians_fixed_kernel (second derivatives with l_max a compile-time number) against the oracle, number for number."""

import numpy as np
import pytest
import torch

from gpu_utils import announce, plan_text, run_launch_layer
from helpers import special_points
from test_gpu_parity import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("normalized", [True, False])
@pytest.mark.parametrize("l_max", range(2, 14))
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_every_l_max(oracle, library, switches, dtype, l_max, normalized):
    """The smallest and largest tile, tiles that are no power of two, one point less and more than a tile, both numbers of
    waves; arrays that start at a multiple of 16 bytes and one element past it, nothing written outside them."""
    if dtype == np.float64 and l_max > (7 if normalized else 10):
        pytest.skip("no kernel")
    ny = (l_max + 1) ** 2
    most = min(32, 160 * 1024 // (13 * (ny + 2) * np.dtype(dtype).itemsize) // 4 * 4)
    for n, tile, waves in ((1, 8, 8), (33, 8, 16), (most - 1, most, 8), (most + 1, most, 16), (50, 12, 8), (263, 20, 16)):
        library.sphx_reset_switches()
        switches("SPHX_HESSIAN_LANES_FIXED", 2)
        switches("SPHX_HESSIAN_LANES_FIXED_TILE", min(tile, most))
        switches("SPHX_HESSIAN_LANES_FIXED_WAVES", waves)
        planned = plan_text(library, n, l_max, "hessians", dtype, normalized)
        name = "double" if dtype == np.float64 else "float"
        assert planned.startswith(f"hessians_fixed_kernel<{name}, {str(normalized).lower()}, {l_max}, {waves}> "
                                  f"[l_max a constant, {min(tile, most)} points"), planned
        xyz = special_points(dtype, np.random.default_rng(l_max), n)
        want = oracle.compute(xyz, l_max, normalized, "hessians")
        for offset in (0, 1):
            announce("second derivatives, l_max a constant", np.dtype(dtype).name, l_max, normalized, n, tile, waves, offset)
            d_xyz = torch.from_numpy(xyz).cuda()
            out = [torch.full((n * c * ny + 2,), -7.0, dtype=d_xyz.dtype, device="cuda") for c in (1, 3, 9)]
            views = tuple(o[offset:offset + n * c * ny] for o, c in zip(out, (1, 3, 9)))
            status, _ = run_launch_layer(library, d_xyz, l_max, normalized, "hessians", out=views)
            torch.cuda.synchronize()
            assert status == 0, library.sphx_last_error()
            check(tuple(v.reshape(w.shape).cpu().numpy() for v, w in zip(views, want)), want, (l_max, n, tile, waves, offset))
            for o in out:
                assert (o[:offset] == -7.0).all() and (o[offset - 2:] == -7.0).all()


@pytest.mark.parametrize("dtype, l_max, n", [(np.float32, 3, 131_072), (np.float32, 4, 9_001), (np.float32, 6, 65_536),
                                             (np.float32, 9, 65_536), (np.float64, 2, 20_000), (np.float64, 5, 65_536),
                                             (np.float64, 7, 1_024), (np.float64, 9, 1_024), (np.float64, 10, 8_192),
                                             (np.float32, 11, 12_287), (np.float32, 12, 4_097), (np.float32, 13, 3_000)])
def test_as_planned(oracle, library, dtype, l_max, n):
    """Calls of sizes between the table's lines, as they are planned."""
    for normalized in (True, False):
        for points in (n - 1, n):
            announce("second derivatives as planned", np.dtype(dtype).name, l_max, normalized, points)
            xyz = special_points(dtype, np.random.default_rng(l_max), points)
            want = oracle.compute(xyz, l_max, normalized, "hessians")
            status, out = run_launch_layer(library, torch.from_numpy(xyz).cuda(), l_max, normalized, "hessians")
            assert status == 0, library.sphx_last_error()
            check(tuple(o.cpu().numpy() for o in out), want, (l_max, points))


@pytest.mark.parametrize("dtype, l_max, normalized, n, below, at", [
    # (kernel<waves> tile, or the kernel without l_max for a constant that is ahead there)
    (np.float32, 3, True, 131_072, "hessians_fixed_kernel<8> 32", "hessians_fixed_kernel<8> 28"),
    (np.float32, 3, False, 131_072, "hessians_fixed_kernel<8> 32", "hessians_fixed_kernel<16> 24"),
    (np.float32, 4, True, 32_768, "hessians_fixed_kernel<16> 32", "hessians_fixed_kernel<8> 32"),
    (np.float32, 6, False, 65_536, "hessians_fixed_kernel<16> 32", "hessians_fixed_kernel<16> 16"),
    (np.float32, 9, True, 65_536, "hessians_fixed_kernel<8> 12", "hessians_fixed_kernel<8> 28"),
    (np.float32, 11, True, 12_288, "hessians_fixed_kernel<8> 20", "recursion_kernel"),
    (np.float32, 12, True, 768, "recursion_kernel", "hessians_fixed_kernel<16> 8"),
    (np.float32, 12, True, 4_097, "hessians_fixed_kernel<16> 16", "recursion_kernel"),
    (np.float32, 13, True, 7_169, "hessians_fixed_kernel<8> 8", "recursion_kernel"),
    (np.float64, 3, False, 65_536, "hessians_fixed_kernel<16> 32", "hessians_fixed_kernel<16> 16"),
    (np.float64, 7, True, 1_024, "recursion_kernel", "hessians_fixed_kernel<8> 8"),
    (np.float64, 9, False, 1_024, "recursion_kernel", "hessians_fixed_kernel<8> 8"),
    (np.float64, 10, False, 8_192, "hessians_fixed_kernel<16> 12", "recursion_kernel"),
    (np.float64, 5, False, 65_536, "hessians_fixed_kernel<16> 24", "hessians_fixed_kernel<16> 16"),
])
def test_both_sides_of_the_tables_lines(oracle, library, dtype, l_max, normalized, n, below, at):
    for points, wanted in ((n - 1, below), (n, at)):
        announce("second derivatives at a line", np.dtype(dtype).name, l_max, normalized, points, wanted)
        planned = plan_text(library, points, l_max, "hessians", dtype, normalized)
        if "_fixed_kernel" in wanted:
            kernel, waves, tile = wanted.replace("<", " ").replace(">", "").split()
            assert planned.startswith(kernel + "<") and f", {l_max}, {waves}> [l_max a constant, {tile} points" in planned, planned
        else:
            assert planned.startswith(wanted + "<"), planned
        xyz = special_points(dtype, np.random.default_rng(l_max), points)
        want = oracle.compute(xyz, l_max, normalized, "hessians")
        status, out = run_launch_layer(library, torch.from_numpy(xyz).cuda(), l_max, normalized, "hessians")
        assert status == 0, library.sphx_last_error()
        check(tuple(o.cpu().numpy() if o is not None else None for o in out), want, (l_max, points))
