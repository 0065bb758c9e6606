"""columns_kernel and column_rows_kernel (sphx_vjp_backward_*, sphx_gradients_backward_*): the second-order products of
a backward pass against the oracle's derivative arrays contracted in float64, and through torch's autograd."""

import numpy as np
import pytest
import torch

import sphericart_amd.torch as sphx_torch
from gpu_utils import announce

pytestmark = pytest.mark.gpu

# Against the oracle in float64 at the same points. From l = 18 on the float32 prefactors underflow (in the reference, too,
# and the kernels use the same ones): there the float32 oracle is the other side. Errors are relative to a point's largest
# sum of absolute terms. The bound: a term has passed through up to l_max steps of a recursion, with a rounding or two
# each, and a tangential derivative is the difference of numbers as large as l times it, in the oracle as here. Hence
# l_max^2 roundings, of 2^-24 or 2^-53, and a few for l_max = 0.
def _tolerance(dtype, l_max):
    return (l_max + 4) ** 2 * np.finfo(dtype).eps / 2


def _cloud(n, dtype, seed):
    rng = np.random.default_rng(seed)
    xyz = rng.standard_normal((n, 3)) + 0.1
    xyz[:: 50, :2] = 0.0  # on the axis
    return xyz.astype(dtype)


def _expected(oracle, xyz, l_max, normalized, w, g, v):
    exact = xyz.astype(np.float64) if l_max <= 17 else xyz
    _, dsph, ddsph = (a.astype(np.float64) for a in oracle.compute(exact, l_max, normalized, "hessians"))
    w, g, v = (a.astype(np.float64) for a in (w, g, v))

    def both(f):
        return f(lambda a: a), f(np.abs)

    hess_w = both(lambda s: np.einsum("iabk,ik,ia->ib", s(ddsph), s(w), s(g)))
    dw = both(lambda s: np.einsum("ia,iak->ik", s(g), s(dsph)))
    hess_v = both(lambda s: np.einsum("iabk,iak->ib", s(ddsph), s(v)))
    grad_w = both(lambda s: np.einsum("iak,ik->ia", s(dsph), s(w)))
    return hess_w, dw, hess_v, grad_w


def _close(got, want, scale, tolerance, what):
    error = np.max(np.abs(got.cpu().numpy().astype(np.float64) - want) / (scale.max(axis=1, keepdims=True) + 1))
    assert error <= tolerance, (what, error)


@pytest.mark.parametrize("tile", [0, 32, 64])
@pytest.mark.parametrize("normalized", [True, False])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_second_order_products_equal_the_oracles_arrays_contracted(library, oracle, dtype, normalized, tile, switches):
    """l_max around the steps that a column's first entries take apart (0-5), odd and even row lengths, the largest each
    kernel holds; points around a tile's 16, 32, 64; both tiles forced where they fit; one wave and eight."""
    suffix = "f32" if dtype == np.float32 else "f64"
    backward, rows = getattr(library, f"sphx_vjp_backward_{suffix}"), getattr(library, f"sphx_gradients_backward_{suffix}")
    stream = torch.cuda.current_stream().cuda_stream
    if tile:
        switches("SPHX_COLUMNS_TILE", tile)
    rng = np.random.default_rng(3)
    for l_max in (0, 1, 2, 3, 4, 5, 6, 7, 9, 12, 16, 17, 24, 25, 26, 27):
        for n, waves in ((1, 0), (15, 8), (33, 1), (65, 3), (700, 0)):
            if waves:
                switches("SPHX_COLUMNS_WAVES", waves)
            announce("second-order products", suffix, normalized, tile, l_max, n, waves)
            if l_max > 12 and n > 100:
                continue
            ny = (l_max + 1) ** 2
            tolerance = _tolerance(dtype, l_max)
            xyz = _cloud(n, dtype, l_max * 100 + n)
            w, g, v = (rng.standard_normal(shape).astype(dtype) for shape in ((n, ny), (n, 3), (n, 3, ny)))
            hess_w, dw, hess_v, grad_w = _expected(oracle, xyz, l_max, normalized, w, g, v)
            d_xyz, d_g, d_v = (torch.from_numpy(a).cuda() for a in (xyz, g, v))
            # the weights once aligned, once one element into a 16-byte vector
            holder = torch.zeros(w.size + 1, dtype=d_xyz.dtype, device="cuda")
            for shift in (0, 1):
                d_w = holder[shift:shift + w.size].view(w.shape)
                d_w.copy_(torch.from_numpy(w))
                out, out_w = torch.full_like(d_xyz, float("nan")), torch.full((n, ny), float("nan"), dtype=d_xyz.dtype, device="cuda")
                status = backward(d_xyz.data_ptr(), d_w.data_ptr(), d_g.data_ptr(), n, l_max, int(normalized), out.data_ptr(),
                                  out_w.data_ptr(), stream)
                if dtype == np.float64 and l_max > 24:
                    assert status == 2
                    continue
                assert status == 0, library.sphx_last_error()
                _close(out, *hess_w, tolerance, (l_max, n, shift, "xyz_grad"))
                _close(out_w, *dw, tolerance, (l_max, n, shift, "sph_grad_grad"))
                for upstream, pointer in ((True, d_w.data_ptr()), (False, None)):
                    out = torch.full_like(d_xyz, float("nan"))
                    status = rows(d_xyz.data_ptr(), pointer, d_v.data_ptr(), n, l_max, int(normalized), out.data_ptr(), stream)
                    if l_max > (24 if dtype == np.float32 else 16):
                        assert status == 2
                        continue
                    assert status == 0, library.sphx_last_error()
                    _close(out, hess_v[0] + upstream * grad_w[0], hess_v[1] + upstream * grad_w[1], tolerance, (l_max, n, shift, upstream))
            if waves:
                switches("SPHX_COLUMNS_WAVES", 0)
    assert backward(None, None, None, 0, 3, 1, None, None, stream) == 0
    assert rows(None, None, None, 0, 3, 1, None, stream) == 0
    assert backward(None, None, None, 5, 3, 1, None, None, stream) == 1


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("l_max", range(1, 22))
def test_kernels_with_l_max_for_a_constant(library, oracle, dtype, l_max, switches):
    """Every l_max that has such a kernel (product 7-20, second-order products 1-12) and the neighbours that do not, both
    parities of the row length; a point less and more than a tile of 16, 32, 64; as planned and with numbers of waves that
    are no power of two or take more vectors per lane than the kernel has under way at a time; weights on and off 16 bytes."""
    suffix = "f32" if dtype == np.float32 else "f64"
    vjp, backward, rows = (getattr(library, f"sphx_{name}_{suffix}") for name in ("vjp", "vjp_backward", "gradients_backward"))
    stream, rng = torch.cuda.current_stream().cuda_stream, np.random.default_rng(l_max)
    ny, tolerance, normalized = (l_max + 1) ** 2, _tolerance(dtype, l_max), l_max % 3 != 0
    for n, waves, tile in ((1, 0, 0), (15, 1, 64), (31, 3, 32), (65, 5, 64), (129, 2, 0)):
        announce("fixed l_max", suffix, l_max, n, waves, tile)
        switches("SPHX_COLUMNS_WAVES", waves)
        switches("SPHX_COLUMNS_TILE", tile)
        xyz = _cloud(n, dtype, n)
        w, g, v = (rng.standard_normal(shape).astype(dtype) for shape in ((n, ny), (n, 3), (n, 3, ny)))
        hess_w, dw, hess_v, grad_w = _expected(oracle, xyz, l_max, normalized, w, g, v)
        d_xyz, d_g = torch.from_numpy(xyz).cuda(), torch.from_numpy(g).cuda()
        w_holder, v_holder = (torch.zeros(a.size + 1, dtype=d_xyz.dtype, device="cuda") for a in (w, v))
        shape = (n, l_max, int(normalized))
        for shift in (0, 1):
            d_w = w_holder[shift:shift + w.size].view(w.shape)
            d_v = v_holder[1 - shift:1 - shift + v.size].view(v.shape)
            d_w.copy_(torch.from_numpy(w))
            d_v.copy_(torch.from_numpy(v))
            out, out_w = torch.full_like(d_xyz, float("nan")), torch.full((n, ny), float("nan"), dtype=d_xyz.dtype, device="cuda")
            assert vjp(d_xyz.data_ptr(), d_w.data_ptr(), *shape, out.data_ptr(), 0, stream) == 0
            _close(out, *grad_w, tolerance, (l_max, n, shift, "product"))
            if l_max > 14:
                continue
            assert backward(d_xyz.data_ptr(), d_w.data_ptr(), d_g.data_ptr(), *shape, out.data_ptr(), out_w.data_ptr(), stream) == 0
            _close(out, *hess_w, tolerance, (l_max, n, shift, "xyz_grad"))
            _close(out_w, *dw, tolerance, (l_max, n, shift, "sph_grad_grad"))
            for upstream, pointer in ((True, d_w.data_ptr()), (False, None)):
                out = torch.full_like(d_xyz, float("nan"))
                assert rows(d_xyz.data_ptr(), pointer, d_v.data_ptr(), *shape, out.data_ptr(), stream) == 0
                _close(out, hess_v[0] + upstream * grad_w[0], hess_v[1] + upstream * grad_w[1], tolerance, (l_max, n, shift, upstream))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_second_order_products_of_large_calls(library, oracle, dtype):
    """The plans of calls with more than 64 points for every CU, as they are made: 64-point tiles and few waves for the
    product's derivatives, the rows' waves by l_max."""
    suffix = "f32" if dtype == np.float32 else "f64"
    backward, rows = getattr(library, f"sphx_vjp_backward_{suffix}"), getattr(library, f"sphx_gradients_backward_{suffix}")
    stream = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(11)
    for l_max, n, normalized in ((1, 40_001, True), (3, 16_390, False), (5, 17_003, True), (6, 33_333, True), (8, 16_401, False), (10, 16_450, True)):
        announce("second-order products, large calls", suffix, l_max, n, normalized)
        ny, tolerance, xyz = (l_max + 1) ** 2, _tolerance(dtype, l_max), _cloud(n, dtype, l_max)
        w, g, v = (rng.standard_normal(shape).astype(dtype) for shape in ((n, ny), (n, 3), (n, 3, ny)))
        hess_w, dw, hess_v, grad_w = _expected(oracle, xyz, l_max, normalized, w, g, v)
        d_xyz, d_w, d_g, d_v = (torch.from_numpy(a).cuda() for a in (xyz, w, g, v))
        out, out_w, out_rows = torch.full_like(d_xyz, float("nan")), torch.full_like(d_w, float("nan")), torch.full_like(d_xyz, float("nan"))
        shape = (n, l_max, int(normalized))
        assert backward(d_xyz.data_ptr(), d_w.data_ptr(), d_g.data_ptr(), *shape, out.data_ptr(), out_w.data_ptr(), stream) == 0
        assert rows(d_xyz.data_ptr(), d_w.data_ptr(), d_v.data_ptr(), *shape, out_rows.data_ptr(), stream) == 0
        _close(out, *hess_w, tolerance, (l_max, n, "xyz_grad"))
        _close(out_w, *dw, tolerance, (l_max, n, "sph_grad_grad"))
        _close(out_rows, hess_v[0] + grad_w[0], hess_v[1] + grad_w[1], tolerance, (l_max, n, "rows"))


def _directions(where, n, seed):
    """Unit vectors on the z axis, within 0.1 of it, or anywhere."""
    rng = np.random.default_rng(seed)
    directions = rng.standard_normal((n, 3))
    if where != "anywhere":
        angle, turn = 0.1 * rng.random(n) * (where == "near"), 2 * np.pi * rng.random(n)
        directions = np.stack([np.sin(angle) * np.cos(turn), np.sin(angle) * np.sin(turn), np.cos(angle)], axis=1)
        directions[:: 2, 2] *= -1
    return directions / np.linalg.norm(directions, axis=1, keepdims=True)


@pytest.mark.parametrize("where", ["axis", "near", "anywhere"])
@pytest.mark.parametrize("normalized", [True, False])
def test_no_further_from_64_bits_than_the_arrays_contracted(library, oracle, normalized, where):
    """float32: the root mean square error of the products over a cloud, each point relative to its largest sum of
    absolute terms, is no larger than that of the float32 derivative arrays contracted in float32, which is what the
    products replace. (Near the z axis a recursion in z alone is 1.4 to 3.8 times that.)"""
    n = 1500
    for l_max in (8, 10, 13, 17):
        announce("error against float64", normalized, where, l_max)
        ny = (l_max + 1) ** 2
        rng = np.random.default_rng(l_max)
        xyz = ((1.0 + rng.random((n, 1))) * _directions(where, n, l_max)).astype(np.float32)
        w, g, v = (rng.standard_normal(shape).astype(np.float32) for shape in ((n, ny), (n, 3), (n, 3, ny)))
        hess_w, dw, hess_v, grad_w = _expected(oracle, xyz, l_max, normalized, w, g, v)
        dsph32 = oracle.compute(xyz, l_max, normalized, "gradients")[1]
        _, dsph, ddsph = oracle.compute(xyz, l_max, normalized, "hessians")
        contracted = {
            "product": np.einsum("iak,ik->ia", dsph32, w),
            "its xyz_grad": np.einsum("iabk,iak->ib", ddsph, g[:, :, None] * w[:, None, :]),
            "its sph_grad_grad": np.einsum("ia,iak->ik", g, dsph),
            "rows": np.einsum("iabk,iak->ib", ddsph, v) + np.einsum("iak,ik->ia", dsph32, w),
        }
        exact = {"product": grad_w, "its xyz_grad": hess_w, "its sph_grad_grad": dw,
                 "rows": (hess_v[0] + grad_w[0], hess_v[1] + grad_w[1])}
        d_xyz, d_w, d_g, d_v = (torch.from_numpy(a).cuda() for a in (xyz, w, g, v))
        product, d_out, rows = (torch.full_like(d_xyz, float("nan")) for _ in range(3))
        d_dw = torch.full_like(d_w, float("nan"))
        stream, shape = torch.cuda.current_stream().cuda_stream, (n, l_max, int(normalized))
        assert library.sphx_vjp_f32(d_xyz.data_ptr(), d_w.data_ptr(), *shape, product.data_ptr(), 0, stream) == 0
        assert library.sphx_vjp_backward_f32(d_xyz.data_ptr(), d_w.data_ptr(), d_g.data_ptr(), *shape, d_out.data_ptr(),
                                             d_dw.data_ptr(), stream) == 0
        assert library.sphx_gradients_backward_f32(d_xyz.data_ptr(), d_w.data_ptr(), d_v.data_ptr(), *shape,
                                                   rows.data_ptr(), stream) == 0
        got = {"product": product, "its xyz_grad": d_out, "its sph_grad_grad": d_dw, "rows": rows}
        for name, (want, scale) in exact.items():
            def error(numbers):
                return np.sqrt(np.mean(((numbers.astype(np.float64) - want) / scale.max(axis=1, keepdims=True)) ** 2))
            here, there = error(got[name].cpu().numpy()), error(contracted[name])
            print(name, here, there, here / there)
            assert here <= there, (name, l_max, here, there)


@pytest.mark.parametrize("tile", [32, 64])
@pytest.mark.parametrize("normalized", [True, False])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_weights_that_are_not_finite_give_what_the_contraction_gives(library, oracle, dtype, normalized, tile, switches):
    """Infinite and NaN weights, upstream gradients and both: every component is the infinity, the NaN or the number that
    adding up the entries' own terms gives; a weight so large that a sum over a column overflows, where no term does,
    gives the finite number; other points of the tile keep theirs bit for bit."""
    suffix = "f32" if dtype == np.float32 else "f64"
    vjp, backward, rows = (getattr(library, f"sphx_{name}_{suffix}") for name in ("vjp", "vjp_backward", "gradients_backward"))
    switches("SPHX_COLUMNS_TILE", tile)
    stream = torch.cuda.current_stream().cuda_stream
    n, l_max = 150, 8
    ny, rng = (l_max + 1) ** 2, np.random.default_rng(5)
    xyz = rng.standard_normal((n, 3))
    xyz = (xyz / np.linalg.norm(xyz, axis=1, keepdims=True) * (1.0 + rng.random((n, 1)))).astype(dtype)
    xyz[100:] *= 20 if normalized else 0.25
    w, g, v = (rng.standard_normal(shape).astype(dtype) for shape in ((n, ny), (n, 3), (n, 3, ny)))

    def run():
        d_xyz, d_w, d_g, d_v = (torch.from_numpy(a).cuda() for a in (xyz, w, g, v))
        first, second, third = (torch.full_like(d_xyz, 7) for _ in range(3))
        dw, shape = torch.full_like(d_w, 7), (n, l_max, int(normalized))
        assert vjp(d_xyz.data_ptr(), d_w.data_ptr(), *shape, first.data_ptr(), 0, stream) == 0
        added = torch.full_like(d_xyz, 7)
        assert vjp(d_xyz.data_ptr(), d_w.data_ptr(), *shape, added.data_ptr(), 1, stream) == 0
        for kind in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(kind(added), kind(first))
        assert backward(d_xyz.data_ptr(), d_w.data_ptr(), d_g.data_ptr(), *shape, second.data_ptr(), dw.data_ptr(), stream) == 0
        assert rows(d_xyz.data_ptr(), d_w.data_ptr(), d_v.data_ptr(), *shape, third.data_ptr(), stream) == 0
        return [t.cpu().numpy() for t in (first, second, dw, third)]

    announce("weights that are not finite", suffix, normalized, tile)
    before = run()
    inf = np.inf
    for i in range(0, 90, 3):  # every third point, an entry of any l and m
        kind, k, a = i // 3 % 6, int(rng.integers(ny)), int(rng.integers(3))
        if kind in (0, 1, 5):
            w[i, k] = inf if kind == 0 else -inf
        if kind in (1, 2):
            v[i, a, k] = -inf
        if kind in (3, 5):
            g[i, a] = inf
        if kind == 4:
            w[i, k] = v[i, a, k] = g[i, a] = np.nan
    with np.errstate(invalid="ignore"):
        _, dsph, ddsph = oracle.compute(xyz, l_max, normalized, "hessians")
        want = [
            (dsph * w[:, None, :]).sum(axis=2),
            (ddsph * (g[:, :, None] * w[:, None, :])[:, :, None, :]).sum(axis=(1, 3)),
            (g[:, :, None] * dsph).sum(axis=1),
            (ddsph * v[:, :, None, :]).sum(axis=(1, 3)) + (dsph * w[:, None, :]).sum(axis=2),
        ]
    after = run()
    for name, got, expected, untouched in zip(("product", "its xyz_grad", "its sph_grad_grad", "rows"), after, want, before):
        for kind in (np.isnan, np.isposinf, np.isneginf):
            np.testing.assert_array_equal(kind(got), kind(expected), err_msg=f"{name} {kind.__name__}")
        rest = np.ones(n, dtype=bool)
        rest[0:90:3] = False
        np.testing.assert_array_equal(got[rest], untouched[rest], err_msg=name)

    # the largest weights there are, at entries whose derivatives are below one: points 100 to 149, far out or close in
    w[:90] = 0
    g[:90] = v[:90] = 1
    most = np.finfo(dtype).max
    for i in range(100, n):
        w[i] = 0
        w[i, int(rng.integers(49, ny))] = most * dtype(0.9)
    first = run()[0]
    exact = (dsph.astype(np.longdouble) * w.astype(np.longdouble)[:, None, :]).sum(axis=2)
    assert (np.abs(exact[100:]) < most).all()
    # one term each: the derivative's own error on either side, _tolerance of the point's largest
    error = np.abs(first[100:] / most - exact[100:] / most).max(axis=1)
    assert (error <= 2 * _tolerance(dtype, l_max) * np.abs(dsph[100:]).max(axis=(1, 2))).all()


@pytest.mark.parametrize("normalized", [True, False])
@pytest.mark.parametrize("l_max", [3, 26])
def test_a_backward_pass_takes_them_and_stays_differentiable(normalized, l_max):
    """Through autograd: the pass without a graph (these kernels; at l_max = 26 the derivative arrays) gives what the
    pass with one (operators that can be differentiated again) gives."""
    announce("second order through autograd", normalized, l_max)
    calculator = (sphx_torch.SphericalHarmonics if normalized else sphx_torch.SolidHarmonics)(l_max)
    torch.manual_seed(2)
    xyz = torch.randn(90, 3, dtype=torch.float64, device="cuda", requires_grad=True)
    w = torch.randn(90, (l_max + 1) ** 2, dtype=torch.float64, device="cuda", requires_grad=True)
    g, v = torch.randn_like(xyz), torch.randn(90, 3, (l_max + 1) ** 2, dtype=torch.float64, device="cuda")
    results = []
    for create_graph in (False, True):
        (forces,) = torch.autograd.grad(calculator(xyz), xyz, w, create_graph=True)
        second = torch.autograd.grad(forces, (xyz, w), g, create_graph=create_graph)
        sph, dsph = calculator.compute_with_gradients(xyz)
        first = torch.autograd.grad((sph, dsph), xyz, (w, v), create_graph=create_graph)
        (only,) = torch.autograd.grad(calculator.compute_with_gradients(xyz)[1], xyz, v, create_graph=create_graph)
        _, dsph, _ = calculator.compute_with_hessians(xyz)
        (third,) = torch.autograd.grad(dsph, xyz, v, create_graph=create_graph)
        results.append((*second, *first, only, third))
        assert all(t.requires_grad == create_graph for t in results[-1])
    for a, b in zip(*results):
        # sums of up to 3 * 729 terms in two orders: 2e-13 of the largest
        assert (a - b).abs().max().item() <= 2e-13 * b.abs().max().item()


@pytest.mark.parametrize("python_operators", ["0", "1"])
def test_a_backward_pass_from_second_derivatives_uses_the_arrays_it_has(python_operators):
    """The pass backward from values, gradients and second derivatives contracts the saved arrays, at an l_max of the
    column kernels and beyond it: number for number, with the points moved in the meantime, and without another array of
    second derivatives."""
    import os
    import subprocess
    import sys

    announce("backward from second derivatives", python_operators)
    code = """
import torch, sphericart_amd.torch
from sphericart_amd.torch import ops as rules
assert rules.cpp_operators == (%r == "0")
ops = torch.ops.sphericart_amd
for l_max in (3, 18):
    for operator in (ops.spherical_harmonics_with_hessians, ops.solid_harmonics_with_hessians):
        torch.manual_seed(l_max)
        xyz = torch.randn(2000, 3, dtype=torch.float64).cuda().requires_grad_()
        sph, dsph, ddsph = operator(xyz, l_max)
        w, v = torch.randn_like(sph), torch.randn_like(dsph)
        with torch.no_grad():
            xyz += 1.0
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        (grad,) = torch.autograd.grad((sph, dsph), xyz, (w, v))
        torch.cuda.synchronize()
        assert torch.cuda.max_memory_allocated() - before < 0.5 * ddsph.numel() * ddsph.element_size(), l_max
        assert torch.equal(grad, ops.contract_gradients(dsph.detach(), w) + ops.contract_hessians(ddsph.detach(), v))
print("done")
""" % python_operators
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=root, timeout=300,
                          env=dict(os.environ, SPHERICART_AMD_PYTHON_OPERATORS=python_operators))
    assert done.returncode == 0 and "done" in done.stdout, done.stderr


def test_which_products_there_are(library):
    """sphx_second_order_supported says what the entries then do."""
    announce("which products")
    for suffix, dtype in (("f32", torch.float32), ("f64", torch.float64)):
        for l_max in (0, 16, 17, 24, 25, 27, 28):
            ny = (l_max + 1) ** 2
            xyz, w, v = (torch.ones(shape, dtype=dtype, device="cuda") for shape in ((5, 3), (5, ny), (5, 3, ny)))
            out, dw = torch.empty_like(xyz), torch.empty_like(w)
            stream, shape = torch.cuda.current_stream().cuda_stream, (5, l_max, 1)
            first = getattr(library, f"sphx_vjp_backward_{suffix}")(
                xyz.data_ptr(), w.data_ptr(), xyz.data_ptr(), *shape, out.data_ptr(), dw.data_ptr(), stream)
            second = getattr(library, f"sphx_gradients_backward_{suffix}")(
                xyz.data_ptr(), w.data_ptr(), v.data_ptr(), *shape, out.data_ptr(), stream)
            for rows, status in ((0, first), (1, second)):
                assert status == (0 if library.sphx_second_order_supported(rows, l_max, int(suffix == "f64")) else 2)
    assert library.sphx_second_order_supported(0, -1, 0) == 0


def test_autograd_with_nothing_but_the_torch_library_loaded(tmp_path):
    """The rules for GPU tensors are in libsphericart_amd_torch.so: a process that has loaded that library alone gets the
    gradients, and the gradients of the gradients, that the package gets."""
    import os
    import subprocess
    import sys

    from sphericart_amd.torch import ops

    announce("autograd, library alone")
    code = f'''
import sys, torch
if sys.argv[1] == "alone":
    torch.ops.load_library({ops.TORCH_LIBRARY_PATH!r})
    assert "sphericart_amd" not in sys.modules
else:
    import sphericart_amd.torch
torch.manual_seed(1)
xyz = torch.randn(77, 3, dtype=torch.float64).cuda().requires_grad_()
w = torch.randn(77, 81, dtype=torch.float64).cuda().requires_grad_()
v = torch.randn(77, 3, 81, dtype=torch.float64).cuda()
ops = torch.ops.sphericart_amd
(forces,) = torch.autograd.grad(ops.spherical_harmonics(xyz, 8), xyz, w, create_graph=True)
out = [forces, *torch.autograd.grad(forces, (xyz, w), torch.ones_like(forces))]
sph, dsph = ops.solid_harmonics_with_gradients(xyz, 8)
out += torch.autograd.grad((sph, dsph), xyz, (w, v))
sph, dsph, ddsph = ops.solid_harmonics_with_hessians(xyz, 8)
out += torch.autograd.grad((sph, dsph), xyz, (w, v))
torch.save([t.detach().cpu() for t in out], sys.argv[2])
'''
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    results = []
    for who in ("alone", "package"):
        path = str(tmp_path / who)
        done = subprocess.run([sys.executable, "-c", code, who, path], capture_output=True, text=True, cwd=root, timeout=300)
        assert done.returncode == 0, done.stderr
        results.append(torch.load(path, weights_only=True))
    for a, b in zip(*results):
        assert torch.equal(a, b)
