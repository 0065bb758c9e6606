"""recursion_kernel with one point per lane (normalised second derivatives in float32, l_max = 4) against the oracle,
number for number."""

import numpy as np
import pytest
import torch

from gpu_utils import announce, plan_text, run_launch_layer
from helpers import special_points
from test_gpu_parity import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("l_max", [4])
@pytest.mark.parametrize("n, forced", [(4096, True), (5003, True), (16383, True), (16384, True), (20011, True), (1_000_003, False)])
@pytest.mark.parametrize("offset", [0, 1])
def test_one_point_per_lane(oracle, library, switches, l_max, n, forced, offset):
    """The smallest calls that have the form (forced; tiles of few points), the smallest for which it is planned, a ragged last
    tile, and outputs that start at an odd element."""
    library.sphx_reset_switches()
    if forced:
        switches("SPHX_POINT_LANES", 1)
    assert plan_text(library, n, l_max, "hessians", np.float32, True).endswith("(one point per lane)")
    ny = (l_max + 1) ** 2
    xyz = special_points(np.float32, np.random.default_rng(67), n)
    want = oracle.compute(xyz, l_max, True, "hessians")
    out = [torch.full((n * c * ny + 2,), -7.0, dtype=torch.float32, device="cuda") for c in (1, 3, 9)]
    views = tuple(o[offset : offset + n * c * ny] for o, c in zip(out, (1, 3, 9)))
    announce("one point per lane", l_max, n, "forced", forced, "offset", offset)
    status, _ = run_launch_layer(library, torch.from_numpy(xyz).cuda(), l_max, True, "hessians", out=views)
    torch.cuda.synchronize()
    assert status == 0, library.sphx_last_error()
    got = tuple(v.reshape(w.shape).cpu().numpy() for v, w in zip(views, want))
    check(got, want, (l_max, n, forced, offset))
    for o in out:  # nothing outside the arrays
        assert (o[:offset] == -7.0).all() and (o[offset - 2 :] == -7.0).all()
    library.sphx_reset_switches()
