"""Calculator classes over the ``sphericart_cuda_*`` C API."""

from typing import Tuple

import torch

from ._c_lib import get_library

# The native handle of a device's current stream: 0.1 us where torch.cuda.current_stream(device).cuda_stream, which makes
# an object of it, takes 1.9.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (
    lambda index: torch.cuda.current_stream(index).cuda_stream)


class _BaseHarmonics:
    # reference: python/src/sphericart/spherical_harmonics.py:9-202
    _cuda_prefix = ""
    _normalized = 0

    def __init__(self, l_max: int, float32_via_float64: bool = False):
        """``float32_via_float64`` (not in the reference, off by default): float32 arrays are
        evaluated in float64 and rounded once (``sphx_forward_f32_via_f64``), which keeps
        l_max >= 29 finite where float32 arithmetic, the reference's included, overflows."""
        if int(l_max) != l_max or l_max < 0:
            raise ValueError("l_max must be a non-negative integer")
        self._l_max = int(l_max)
        self._float32_via_float64 = bool(float32_via_float64)
        self._lib = get_library()
        self._calculator_cuda = None
        self._calculator_cuda_f = None
        self._functions = None  # by dtype: the calculator and its three functions

    def __del__(self):
        self._delete_calculator(f"{self._cuda_prefix}_delete", "_calculator_cuda")
        self._delete_calculator(f"{self._cuda_prefix}_delete_f", "_calculator_cuda_f")

    def _delete_calculator(self, function_name: str, attribute: str):
        calculator = getattr(self, attribute, None)
        if calculator is not None:
            getattr(self._lib, function_name)(calculator)
            setattr(self, attribute, None)

    def _validate_xyz(self, xyz):
        if not isinstance(xyz, torch.Tensor):
            raise TypeError("xyz must be a torch.Tensor on a ROCm device")
        if xyz.dtype not in (torch.float32, torch.float64):
            raise TypeError("xyz must be an array of 32 or 64-bit floats")
        if xyz.dim() != 2 or xyz.shape[1] != 3:
            raise ValueError("xyz array must be a `N x 3` array")
        if not xyz.is_cuda:
            raise ValueError(
                "xyz must live on a ROCm device: sphericart_amd has no CPU evaluation path"
            )
        return xyz.contiguous()

    def _ensure_cuda_calculators(self):
        if self._functions is not None:
            return
        self._calculator_cuda = getattr(self._lib, f"{self._cuda_prefix}_new")(self._l_max)
        self._calculator_cuda_f = getattr(self._lib, f"{self._cuda_prefix}_new_f")(self._l_max)
        if self._calculator_cuda and self._calculator_cuda_f:
            names = [f"{self._cuda_prefix}_compute_array{what}" for what in ("", "_with_gradients", "_with_hessians")]
            self._functions = {
                torch.float64: (self._calculator_cuda, *(getattr(self._lib, name) for name in names)),
                torch.float32: (self._calculator_cuda_f, *(getattr(self._lib, name + "_f") for name in names)),
            }
            return
        self._delete_calculator(f"{self._cuda_prefix}_delete", "_calculator_cuda")
        self._delete_calculator(f"{self._cuda_prefix}_delete_f", "_calculator_cuda_f")
        raise RuntimeError(
            "failed to initialize the device calculators; a HIP device must be visible and "
            "l_max must not exceed what the device tables cover"
        )

    def _compute_impl(self, xyz, gradients: bool = False, hessians: bool = False):
        xyz = self._validate_xyz(xyz)
        self._ensure_cuda_calculators()

        n_samples = xyz.shape[0]
        lmtotal = (self._l_max + 1) ** 2
        if type(xyz) is torch.Tensor:  # (what a call costs the host: 1.4 us per array, 1.7 from torch.empty)
            empty = xyz.new_empty
        else:
            def empty(shape):
                return torch.empty(shape, dtype=xyz.dtype, device=xyz.device)
        sph = empty((n_samples, lmtotal))
        dsph = empty((n_samples, 3, lmtotal)) if gradients else None
        ddsph = empty((n_samples, 3, 3, lmtotal)) if hessians else None

        if self._float32_via_float64 and xyz.dtype == torch.float32 and n_samples > 0:
            self._compute_via_float64(xyz, sph, dsph, ddsph)
            return (sph, dsph, ddsph) if hessians else (sph, dsph) if gradients else sph

        # (the library takes the device from the xyz pointer: no need to make it current here)
        stream = _raw_stream(xyz.get_device())
        calculator, values, with_gradients, with_hessians = self._functions[xyz.dtype]
        if hessians:
            with_hessians(calculator, xyz.data_ptr(), n_samples, sph.data_ptr(), dsph.data_ptr(), ddsph.data_ptr(), stream)
            return sph, dsph, ddsph
        if gradients:
            with_gradients(calculator, xyz.data_ptr(), n_samples, sph.data_ptr(), dsph.data_ptr(), stream)
            return sph, dsph
        values(calculator, xyz.data_ptr(), n_samples, sph.data_ptr(), stream)
        return sph

    def _compute_via_float64(self, xyz, sph, dsph, ddsph):
        derivatives = 2 if ddsph is not None else (1 if dsph is not None else 0)
        n_samples = xyz.shape[0]
        # Beyond the closed forms the library evaluates in one launch and needs no workspace (if a
        # shape should not fit that launch it takes one from the device's pool, in stream order).
        # Below, a workspace from torch's allocator: at most 256 MiB, the library walks over the
        # points in chunks of what it holds.
        workspace, size = None, 0
        if self._l_max <= (1 if derivatives == 2 else 6):
            wanted = self._lib.sphx_forward_f32_via_f64_workspace(n_samples, self._l_max, derivatives)
            floor = self._lib.sphx_forward_f32_via_f64_workspace(min(n_samples, 64), self._l_max, derivatives)
            size = max(min(wanted, 256 << 20), floor)
            workspace = torch.empty(size, dtype=torch.uint8, device=xyz.device)
        with torch.cuda.device(xyz.device):
            stream = torch.cuda.current_stream()
            status = self._lib.sphx_forward_f32_via_f64(
                xyz.data_ptr(), n_samples, self._l_max, self._normalized, derivatives,
                sph.data_ptr(), dsph.data_ptr() if dsph is not None else None,
                ddsph.data_ptr() if ddsph is not None else None,
                workspace.data_ptr() if workspace is not None else None, size, stream.cuda_stream,
            )
            if workspace is not None:
                workspace.record_stream(stream)
        if status != 0:
            raise RuntimeError(self._lib.sphx_last_error().decode())

    def compute(self, xyz):
        """Values, ``(n_samples, (l_max+1)**2)``."""
        return self._compute_impl(xyz)

    def compute_with_gradients(self, xyz) -> Tuple[torch.Tensor, torch.Tensor]:
        """Values and Cartesian gradients, ``(n_samples, 3, (l_max+1)**2)``."""
        return self._compute_impl(xyz, gradients=True)

    def compute_with_hessians(self, xyz) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
        """Values, gradients and Hessians, ``(n_samples, 3, 3, (l_max+1)**2)``."""
        return self._compute_impl(xyz, gradients=True, hessians=True)


class SphericalHarmonics(_BaseHarmonics):
    """Real spherical harmonics :math:`Y^m_l` up to ``l_max`` of points given in Cartesian coordinates."""

    _cuda_prefix = "sphericart_cuda_spherical_harmonics"
    _normalized = 1


class SolidHarmonics(_BaseHarmonics):
    """Solid harmonics :math:`r^l Y^m_l` up to ``l_max``."""

    _cuda_prefix = "sphericart_cuda_solid_harmonics"
