"""The work a user of sphericart_amd has it do, as a list of cases and a generator of more of the same ranges.

``listed()`` names the cases, ``draw(rng)`` makes another one, ``prepare`` builds what a program holds before the call
(a calculator or module and its tensors on the GPU), ``run`` is one pass through the public entry points, ``work``
counts the bytes and operations a pass cannot do without and ``tolerance`` says how far another correct implementation
in the same precision would be off.

A case has the fields

``kind``       what is computed:
               ``values``, ``gradients``, ``hessians``: a forward evaluation;
               ``train``: values, then the vector-Jacobian product (``sph`` enters a model, the model's
               gradient comes back to the coordinates);
               ``forces``: a model trained on forces: values, forces as the vector-Jacobian product with the graph
               kept, then the backward pass through the forces to the coordinates and the model's weights;
               ``derivatives``: values and gradients as a model's features, then the backward pass from both.
``entry``      ``calculator`` (``sphericart_amd.SphericalHarmonics`` / ``SolidHarmonics``, the ``sphericart_cuda_*``
               API) or ``module`` (``sphericart_amd.torch``); the kinds with a backward pass need the module.
``harmonics``  ``spherical`` or ``solid``.
``dtype``      ``float32`` or ``float64``.
``l_max``, ``n``  order and number of points.
``cloud``      how the points lie: ``shell`` (uniform directions, radii 0.5 to 5, neighbour vectors within a cutoff),
               ``normal`` (bell-shaped coordinates), ``box`` (uniform in [-3, 3)^3), ``octaves`` (radii from 0.01 to 82,
               the same share in each octave). One point in a hundred of ``shell`` and ``octaves`` is on the z axis.
"""

import math

import torch

import sphericart_amd
import sphericart_amd.torch


def _case(name, kind, entry, harmonics, dtype, l_max, n, cloud):
    case = {"kind": kind, "entry": entry, "harmonics": harmonics, "dtype": dtype, "l_max": l_max, "n": n, "cloud": cloud}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one small molecule's pairs at inference: launches and host time are all there is
        _case("molecule values", "values", "module", "spherical", "float32", 4, 300, "shell"),
        # a training step on one small structure: forward and backward, still bound by latency
        _case("molecule training step", "train", "module", "spherical", "float32", 6, 1500, "shell"),
        # the benchmark's configurations, from the small double precision call to the largest arrays
        _case("l8 f64 gradients 10k", "gradients", "calculator", "spherical", "float64", 8, 10_000, "normal"),
        _case("l3 f32 values 1M", "values", "calculator", "spherical", "float32", 3, 1_000_000, "shell"),
        _case("l6 f32 gradients 1M", "gradients", "calculator", "spherical", "float32", 6, 1_000_000, "shell"),
        _case("l16 f64 solid hessians 100k", "hessians", "calculator", "solid", "float64", 16, 100_000, "box"),
        _case("l32 f32 gradients 200k", "gradients", "calculator", "spherical", "float32", 32, 200_000, "octaves"),
        # values alone far beyond the closed forms
        _case("l22 f32 values 500k", "values", "calculator", "spherical", "float32", 22, 500_000, "shell"),
        # second derivatives at the orders interatomic potentials use
        _case("l5 f32 hessians 500k", "hessians", "calculator", "spherical", "float32", 5, 500_000, "shell"),
        # a training step on a large batch of structures (a ragged number of pairs)
        _case("l8 f32 training step 400k", "train", "module", "spherical", "float32", 8, 400_003, "shell"),
        # training on forces: the pass backward through a backward pass
        _case("l6 f32 force training 120k", "forces", "module", "spherical", "float32", 6, 120_000, "shell"),
        # gradients as features in double precision, trained through
        _case("l9 f64 solid derivatives 20k", "derivatives", "module", "solid", "float64", 9, 20_011, "shell"),
    ]


_KINDS = ("values", "gradients", "hessians", "train", "forces", "derivatives")
# the largest l_max a kind is asked for
_TOP = {"values": 32, "gradients": 32, "hessians": 20, "train": 20, "forces": 12, "derivatives": 12}
# numbers moved per point and component of a row, for the bound on a drawn case's size
_SPREAD = {"values": 1, "gradients": 4, "hessians": 13, "train": 8, "forces": 40, "derivatives": 32}
_LARGEST = 2.5e9  # bytes


def draw(rng):
    kind = rng.choice(_KINDS)
    dtype = rng.choice(("float32", "float64"))
    l_max = rng.randint(1, _TOP[kind])
    size = 4 if dtype == "float32" else 8
    most = min(1_000_000, int(_LARGEST / (size * _SPREAD[kind] * (l_max + 1) ** 2)))
    n = int(math.exp(rng.uniform(math.log(200), math.log(most))))
    entry = rng.choice(("calculator", "module")) if kind in ("values", "gradients", "hessians") else "module"
    harmonics = rng.choice(("spherical", "solid"))
    cloud = rng.choice(("shell", "normal"))
    return _case(None, kind, entry, harmonics, dtype, l_max, n, cloud)


def _points(case, dtype, random):
    n, cloud = case["n"], case["cloud"]

    def uniform(*shape):
        return torch.rand(*shape, dtype=torch.float64, device="cuda", generator=random)

    def normal(*shape):
        return torch.randn(*shape, dtype=torch.float64, device="cuda", generator=random)

    if cloud == "normal":
        return normal(n, 3).to(dtype)
    if cloud == "box":
        return (6.0 * uniform(n, 3) - 3.0).to(dtype)
    if cloud == "shell":
        radius = 0.5 + 4.5 * uniform(n, 1)
    else:
        radius = 0.01 * torch.exp2(torch.floor(13.0 * uniform(n, 1))) * (1.0 + uniform(n, 1))
    direction = normal(n, 3)
    direction[::100, :2] = 0.0
    direction = direction / direction.norm(dim=1, keepdim=True)
    return (radius * direction).to(dtype)


def prepare(case, seed):
    random = torch.Generator(device="cuda")
    random.manual_seed(int(seed))
    dtype = getattr(torch, case["dtype"])
    kind, n, row = case["kind"], case["n"], (case["l_max"] + 1) ** 2
    classes = sphericart_amd if case["entry"] == "calculator" else sphericart_amd.torch
    cls = classes.SphericalHarmonics if case["harmonics"] == "spherical" else classes.SolidHarmonics

    def weights(*shape):
        return torch.randn(*shape, dtype=dtype, device="cuda", generator=random)

    state = {"kind": kind, "calculator": cls(case["l_max"]), "xyz": _points(case, dtype, random)}
    if kind in ("train", "forces", "derivatives"):
        state["xyz"].requires_grad_(True)
        state["sph_grad"] = weights(n, row)  # what the model hands back
    if kind == "forces":
        state["sph_grad"].requires_grad_(True)
        state["force_grad"] = weights(n, 3)
    if kind == "derivatives":
        state["dsph_grad"] = weights(n, 3, row)
    return state


def run(state):
    kind, calculator, xyz = state["kind"], state["calculator"], state["xyz"]
    if kind == "values":
        return calculator.compute(xyz)
    if kind == "gradients":
        return calculator.compute_with_gradients(xyz)
    if kind == "hessians":
        return calculator.compute_with_hessians(xyz)
    if kind == "train":
        sph = calculator(xyz)
        (xyz_grad,) = torch.autograd.grad(sph, xyz, state["sph_grad"])
        return sph.detach(), xyz_grad
    if kind == "forces":
        sph = calculator(xyz)
        (forces,) = torch.autograd.grad(sph, xyz, state["sph_grad"], create_graph=True)
        xyz_grad, sph_grad_grad = torch.autograd.grad(forces, (xyz, state["sph_grad"]), state["force_grad"])
        return sph.detach(), forces.detach(), xyz_grad, sph_grad_grad
    sph, dsph = calculator.compute_with_gradients(xyz)
    (xyz_grad,) = torch.autograd.grad((sph, dsph), xyz, (state["sph_grad"], state["dsph_grad"]))
    return sph.detach(), dsph.detach(), xyz_grad


def work(case):
    """Each input of each call read once and each output written once; operations of the recursion, the prefactors
    and the chain rule per component, and two per term of a contraction."""
    n, row = case["n"], (case["l_max"] + 1) ** 2
    size = 4 if case["dtype"] == "float32" else 8
    numbers, operations = {
        "values": (3 + row, 4 * row),
        "gradients": (3 + 4 * row, 20 * row),
        "hessians": (3 + 13 * row, 80 * row),
        "train": (3 + row + 3 + row + 3, (4 + 20 + 6) * row),
        "forces": (3 + row + 3 + row + 3 + 3 + row + 3 + 3 + row, (4 + 20 + 6 + 80 + 18) * row),
        "derivatives": (3 + 4 * row + 3 + 4 * row + 3, (20 + 80 + 24) * row),
    }[case["kind"]]
    return {"bytes": size * n * numbers, "flops": n * operations}


def tolerance(case):
    """Float32 against the same calls in float64, over these ranges up to l_max = 17 (from about 20 on float32 itself
    underflows, in every implementation of the recursion): at most 1e-6 relative and 1.3e-4 in one number. Float64
    with the sums of the contractions reversed and the low orders by recursion instead of in closed form: at most
    6.4e-15 and 1.7e-13. About four times that."""
    if case["dtype"] == "float32":
        return {"rel": 5e-6, "max": 5e-4}
    return {"rel": 3e-14, "max": 1e-12}
