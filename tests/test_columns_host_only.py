"""The planner of the column kernels is plain host C++ (sphx_columns.cpp with sphx_plan.cpp, compiled with g++ alone): which
kernel a vector-Jacobian product gets, and that what is planned fits."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sphericart_amd", "csrc")
VJP, VJP_BACKWARD, ROWS = 0, 1, 2


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    binary = tmp_path_factory.mktemp("columns") / "columns_probe"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", os.path.join(ROOT, "tests", "columns_probe.cpp"),
                    *(os.path.join(CSRC, name) for name in ("sphx_columns.cpp", "sphx_plan.cpp")), "-o", str(binary)], check=True)

    def run(shapes, **switches):
        """`switches`: overrides, read from the environment under SPHX_DEBUG_SWITCHES."""
        names = "there groups workgroups threads lds tiles pad off_rows off_sums by_columns fixed".split()
        env = dict(os.environ, SPHX_DEBUG_SWITCHES="1", **{name: str(value) for name, value in switches.items()})
        out = subprocess.run([str(binary)] + [str(v) for shape in shapes for v in shape], capture_output=True, text=True,
                             check=True, env=env).stdout.splitlines()
        assert len(out) == len(shapes)
        return [dict(zip(names, map(int, line.split()))) for line in out]

    return run


def test_which_kernel_a_product_gets(plans):
    """The columns beyond the closed forms, but where the lane kernel takes a round less (float64 from l_max = 17, float32
    at 20 and from 25), up to four rounds."""
    wanted = {
        (1_000, 6, 4): False, (1_000, 7, 4): True, (400_003, 8, 4): True, (1_500, 24, 8): True, (1_500, 25, 8): False,
        (1_500, 27, 4): True, (1_500, 28, 4): False,
        (8_000, 17, 8): True, (9_000, 17, 8): False, (15_000, 17, 8): True, (17_000, 17, 8): False, (41_100, 17, 8): False,
        (200_000, 17, 8): True, (9_000, 18, 8): False, (9_000, 19, 8): False, (9_000, 20, 8): True, (9_000, 16, 8): True,
        (17_600, 20, 4): False, (19_000, 20, 4): True, (17_600, 19, 4): True, (9_000, 24, 4): True, (9_000, 25, 4): False,
        (15_000, 26, 4): True, (41_100, 26, 4): False, (200_000, 26, 4): True,
    }
    for shape, plan in zip(wanted, plans([(VJP, *shape) for shape in wanted])):
        assert bool(plan["by_columns"]) == wanted[shape], shape


@pytest.mark.parametrize("elem", [4, 8])
def test_which_products_have_a_kernel_with_l_max_for_a_constant(plans, elem):
    """The product at l_max = 7-20, the second-order ones at 1-12, on two lanes per point and, where three tiles of 64 points
    fit a CU, on one; calls of every size, and the settings that tests/test_gpu_columns.py forces on small ones."""
    first_last = {VJP: (7, 20), VJP_BACKWARD: (1, 12), ROWS: (1, 12)}
    for waves, tile, points in ((0, 0, (1, 129, 16_384, 16_385, 400_003)), (1, 64, (15,)), (3, 32, (31,)), (5, 64, (65,)), (2, 0, (129,))):
        shapes = [(kind, n, l_max, elem) for kind in first_last for l_max in range(28) for n in points]
        for (kind, n, l_max, _), plan in zip(shapes, plans(shapes, SPHX_COLUMNS_WAVES=waves, SPHX_COLUMNS_TILE=tile)):
            ny = (l_max + 1) ** 2
            row = (ny + (1 if ny % 2 == 0 and ny > 16 // elem else 0)) * elem
            lanes = kind == ROWS or plan["groups"] == 2 or 3 * 64 * row <= 160 * 1024
            wanted = plan["there"] and first_last[kind][0] <= l_max <= first_last[kind][1] and lanes
            assert bool(plan["fixed"]) == bool(wanted), (kind, n, l_max, waves, tile)
            if l_max <= 6 and tile == 64 and kind != ROWS:
                assert plan["groups"] == 1 and plan["fixed"] == (kind == VJP_BACKWARD and l_max > 0)


@pytest.mark.parametrize("elem", [4, 8])
def test_what_is_planned_fits(plans, elem):
    """Rows, pads and the sums of the waves inside LDS, tiles for all points, at most 512 threads and fewer than 2^32 in a
    launch; and where the tables or LDS end there is no plan."""
    reach = {VJP: 27 if elem == 4 else 24, VJP_BACKWARD: 27 if elem == 4 else 24, ROWS: 24 if elem == 4 else 16}
    shapes = [(kind, n, l_max, elem) for kind in reach for l_max in range(31)
              for n in (1, 15, 1_000, 16_384, 16_385, 400_003, 30_000_000, 600_000_000, 1_200_000_000, 5_000_000_000)]
    for (kind, n, l_max, _), plan in zip(shapes, plans(shapes)):
        if l_max > reach[kind]:
            assert not plan["there"], (kind, n, l_max)
            continue
        if not plan["there"]:  # one wave per tile is too many already
            assert n > 2**32 // (64 // (16 if kind == ROWS else 32)) - 1_000, (kind, n, l_max)
            continue
        assert plan["threads"] % 64 == 0 and 64 <= plan["threads"] <= 512
        assert plan["workgroups"] % 8 == 0 and plan["workgroups"] * plan["threads"] < 2**32, (kind, n, l_max)
        tile = 64 // plan["groups"]
        assert plan["groups"] in ((4,) if kind == ROWS else (1, 2))
        assert (plan["tiles"] - 1) * tile < n <= plan["tiles"] * tile and plan["workgroups"] >= plan["tiles"]
        ny, waves = (l_max + 1) ** 2, plan["threads"] // 64
        assert plan["pad"] in (0, 1) and (plan["pad"] == 0 or ny % (16 // elem) == 0)
        rows = plan["off_rows"] + tile * (ny + plan["pad"])
        assert kind != ROWS or plan["off_rows"] >= tile * (3 * ny + plan["pad"])
        sums = (waves - 1) * (7 * 16 if kind == ROWS else (3 if kind == VJP else 6) * 64)
        assert kind != VJP_BACKWARD or plan["off_sums"] >= rows
        assert max(rows, plan["off_sums"] + sums) * elem <= plan["lds"] <= 160 * 1024
