"""The planner is plain host C++: sphx_plan.cpp compiles with g++ alone (no HIP header, no device) into a small
program, whose plans for a spread of shapes are those the library reports through sphx_describe_plan, word for
word, and name the kernels the shapes are meant to get."""

import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sphericart_amd", "csrc")

SHAPES = [
    # n_samples, l_max, mode, is_f64, normalized, the kernel it is meant to get
    (1_000_000, 6, 1, 0, 1, "gradients_lanes_kernel<float, true>"),
    (1_000_000, 3, 0, 0, 1, "closed_form_kernel<float, 0, true, 3, false>"),
    (10_000, 8, 1, 1, 1, "gradients_fixed_kernel<double, true, 8, 8>"),
    (100_000, 16, 2, 1, 0, "recursion_kernel<double, 2, false, true, true, false, true>"),
    (200_000, 32, 1, 0, 1, "pairs_kernel<float, 1, true>"),
    (200_000, 32, 0, 0, 1, "values_fixed_kernel<float, true, 32, 8>"),
    (200_000, 34, 0, 0, 1, "pairs_kernel<float, 0, true>"),
    (200_000, 20, 0, 1, 0, "values_fixed_kernel<double, false, 20, 8>"),
    (200_000, 25, 0, 1, 0, "pairs_kernel<double, 0, false>"),
    (1_000_000, 10, 0, 0, 1, "values_kernel<float, true, 1>"),
    (3_000_000, 9, 0, 0, 1, "values_kernel<float, true, 1>"),
    (1_000_000, 22, 0, 0, 1, "values_fixed_kernel<float, true, 22, 8>"),
    (1_000_000, 13, 0, 0, 1, "values_kernel<float, true, 2>"),
    (100_000, 8, 0, 0, 1, "values_fixed_kernel<float, true, 8, 4>"),
    (3_500_000, 8, 0, 0, 0, "values_fixed_kernel<float, false, 8, 4>"),
    (300_000, 22, 0, 0, 1, "values_fixed_kernel<float, true, 22, 8>"),
    (500_000, 22, 0, 0, 0, "values_fixed_kernel<float, false, 22, 8>"),
    (100_000, 4, 2, 0, 1, "hessians_fixed_kernel<float, true, 4, 8>"),
    (600_000, 4, 2, 0, 1, "hessians_fixed_kernel<float, true, 4, 8>"),
    (500_000, 5, 2, 0, 1, "hessians_fixed_kernel<float, true, 5, 16>"),
    (1_000_000, 4, 2, 0, 1, "recursion_kernel<float, 2, true, true, false, false, true>"),
    (500_000, 3, 2, 0, 1, "hessians_fixed_kernel<float, true, 3, 8>"),
    (4_000_000, 2, 2, 0, 1, "hessians_lanes_kernel<float, true>"),
    (1_000_000, 7, 0, 0, 0, "values_fixed_kernel<float, false, 7, 4>"),
    (2_000, 5, 2, 0, 1, "hessians_fixed_kernel<float, true, 5, 16>"),
    (600_000, 7, 1, 0, 0, "gradients_lanes_kernel<float, false>"),
    (1_000_000, 10, 1, 0, 1, "gradients_fixed_kernel<float, true, 10, 16>"),
    (1_000_000, 10, 1, 0, 0, "recursion_kernel<float, 1, false, true, false, false, true>"),
    (100_000, 19, 1, 0, 1, "recursion_kernel<float, 1, true, true, false, false, true>"),
    (50_000, 20, 2, 1, 1, "pairs_kernel<double, 2, true>"),
    (2_000, 32, 1, 0, 1, "recursion_kernel<float, 1, true, true, false, false, true>"),
    (2_000, 40, 1, 1, 1, "recursion_kernel<double, 1, true, false, false, false, false>"),
    (5, 24, 2, 1, 1, "recursion_kernel<double, 2, true, true, false, false, false>"),
    (1, 0, 0, 0, 1, "closed_form_kernel<float, 0, true, 0, false>"),
    # values: channels side by side, four or eight by the rounds that the tiles take on the CUs
    (600_000, 16, 0, 0, 1, "values_kernel<float, true, 2>"),
    (300_000, 17, 0, 0, 1, "values_kernel<float, true, 4>"),
    (1_000_000, 10, 0, 1, 1, "values_kernel<double, true, 1>"),
    (500_000, 14, 0, 1, 1, "values_kernel<double, true, 2>"),
    (9_000, 29, 0, 1, 1, "values_kernel<double, true, 4>"),
    (4_000, 33, 0, 0, 1, "values_kernel<float, true, 4>"),
    (9_000, 33, 0, 0, 1, "values_kernel<float, true, 8>"),
    # values and second derivatives in mid-sized and large calls: no gaps between the ranges
    (60_000, 12, 0, 0, 1, "values_fixed_kernel<float, true, 12, 8>"),
    (12_000, 26, 0, 0, 1, "values_fixed_kernel<float, true, 26, 8>"),
    (20_000, 28, 0, 0, 1, "values_fixed_kernel<float, true, 28, 8>"),
    (1_000_000, 30, 0, 0, 1, "values_fixed_kernel<float, true, 30, 8>"),
    (10_000, 18, 0, 1, 1, "values_fixed_kernel<double, true, 18, 8>"),
    (9_000, 21, 0, 1, 1, "values_fixed_kernel<double, true, 21, 8>"),
    (20_000, 23, 0, 1, 1, "values_fixed_kernel<double, true, 23, 8>"),
    (2_000_000, 10, 1, 0, 1, "gradients_fixed_kernel<float, true, 10, 16>"),
    # the flush at raised priority: by the table of shapes, and only with many tiles per workgroup
    (200_000, 33, 1, 0, 0, "pairs_kernel<float, 1, false>"),
    (40_000, 33, 1, 0, 0, "pairs_kernel<float, 1, false>"),
    (300_000, 10, 2, 0, 0, "recursion_kernel<float, 2, false, true, false, false, true>"),
    (300_000, 9, 2, 0, 0, "recursion_kernel<float, 2, false, true, false, false, true>"),
    (300_000, 14, 2, 0, 0, "recursion_kernel<float, 2, false, true, false, false, true>"),
    (300_000, 15, 2, 0, 0, "recursion_kernel<float, 2, false, true, false, false, true>"),
]
PRIORITY = {(200_000, 33, 1, 0): True, (300_000, 14, 2, 0): True, (300_000, 10, 2, 0): True, (1_000_000, 10, 1, 0): True}  # (n, l_max, mode, normalized)


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    binary = tmp_path_factory.mktemp("planner") / "planner_probe"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", os.path.join(ROOT, "tests", "planner_probe.cpp"),
                    os.path.join(CSRC, "sphx_plan.cpp"), "-o", str(binary)], check=True)
    return str(binary)


def test_plans_without_a_device_match_the_library_and_name_the_intended_kernels(probe, library):
    args = [str(v) for shape in SHAPES for v in shape[:5]]
    lines = subprocess.run([probe] + args, capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(lines) == len(SHAPES)
    library.sphx_reset_switches()
    for (n, l_max, mode, is_f64, normalized, kernel), line in zip(SHAPES, lines):
        text = ctypes.create_string_buffer(1024)
        assert library.sphx_describe_plan(n, l_max, mode, is_f64, normalized, text, len(text)) == 0
        assert line == text.value.decode(), (n, l_max, mode, is_f64, normalized)
        assert line.split(" + ")[-1].startswith(kernel + " ["), (line, kernel)
        assert line.endswith("(flush at raised priority)") == PRIORITY.get((n, l_max, mode, normalized), False), line


def test_every_row_of_the_planners_tables_is_reached(tmp_path):
    """No row, and no l_max of one, that no call is planned by: such a row is a figure nobody can check by calling."""
    binary = tmp_path / "rows_probe"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", os.path.join(ROOT, "tests", "rows_probe.cpp"),
                    *(os.path.join(CSRC, name) for name in ("sphx_plan.cpp", "sphx_columns.cpp")), "-o", str(binary)], check=True)
    out = subprocess.run([str(binary)], capture_output=True, text=True, check=True).stdout.splitlines()
    assert out == ["done"], out


def test_shapes_beyond_the_tables_or_lds_are_refused_with_a_message(probe):
    out = subprocess.run([probe, "10", "65", "0", "0", "1", "10", "64", "2", "1", "1"], capture_output=True, text=True,
                         check=True).stdout.splitlines()
    assert out[0].startswith("status 2:") and "prefactor tables" in out[0]
    assert out[1].startswith("status 2:") and "LDS" in out[1]
