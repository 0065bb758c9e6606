"""The Python calculators' call: the stream it goes to, and tensors that are not plain ones."""

import numpy as np
import pytest
import torch

import sphericart_amd
from gpu_utils import METHOD, announce
from helpers import same_numbers

pytestmark = pytest.mark.gpu


class _Named(torch.Tensor):
    pass


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("mode", ["values", "gradients", "hessians"])
def test_goes_to_the_current_stream_and_returns_plain_tensors(oracle, mode, dtype):
    """The coordinates are written on a side stream behind a long wait: a call that went anywhere else would read the zeros
    before them. Parameters, tensors of a subclass and slices that are not contiguous give plain arrays without a gradient."""
    calculator = sphericart_amd.SphericalHarmonics(5)
    host = torch.from_numpy(np.random.default_rng(2).standard_normal((211, 3))).to(dtype)
    want = oracle.compute(host.numpy(), 5, True, mode)
    announce("calculators", mode, dtype)
    ready, xyz, side = host.cuda(), torch.zeros(211, 3, dtype=dtype, device="cuda"), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
        xyz.copy_(ready)
        first = getattr(calculator, METHOD[mode])(xyz)
    side.synchronize()
    strided = torch.zeros(211, 6, dtype=dtype, device="cuda")
    strided[:, ::2] = ready
    for out in (first, *(getattr(calculator, METHOD[mode])(x) for x in (torch.nn.Parameter(ready), ready.as_subclass(_Named), strided[:, ::2]))):
        for got, expected in zip((out,) if mode == "values" else out, want):
            assert type(got) is torch.Tensor and not got.requires_grad
            assert same_numbers(got.cpu().numpy(), expected).all()
