"""PolarQuant with the reference's interface (turboquant/polar_quant.py:46-132):
norm extraction, rotation, nearest Lloyd-Max centroid per coordinate.

Tables are built on the host exactly as the reference builds them; quantize,
dequantize and the residual run as float64 HIP kernels (tq_quantize_indices,
tq_dequantize_indices).  `rotation="wht"` replaces the dense Haar rotation by
the sign-diagonal Walsh-Hadamard rotation D2 H D1 (signs drawn from the same
seeded generator as turboquant/rotation.py:94-95).
"""
from __future__ import annotations

import numpy as np

from . import _lib as L
from .codebook import optimal_centroids
from .rotation import random_rotation_dense, random_rotation_fast


class PolarQuant:
    def __init__(self, d: int, bit_width: int, seed: int = 42, norm_correction: bool = True, *,
                 rotation: str = "dense"):
        if rotation not in ("dense", "wht"):
            raise ValueError(f"rotation must be 'dense' or 'wht', got {rotation!r}")
        if not 1 <= bit_width <= 8:
            raise ValueError(f"bit_width must be 1-8, got {bit_width}")
        self.d = d
        self.bit_width = bit_width
        self.n_centroids = 1 << bit_width
        self.norm_correction = norm_correction
        self.rotation_mode = rotation
        rng = np.random.default_rng(seed)
        if rotation == "dense":
            self.rotation = random_rotation_dense(d, rng)
            self.signs1 = self.signs2 = None
        else:
            self.signs1, self.signs2, self.padded_d = random_rotation_fast(d, rng)
            self.rotation = None
        self.centroids = optimal_centroids(bit_width, d)
        self._handle = None

    # the device tables are created on first use so that constructing a
    # quantiser (and reading .rotation / .centroids) needs no GPU
    @property
    def handle(self) -> L.Handle:
        if self._handle is None:
            self._handle = L.Handle(self.d, self.bit_width, self.centroids, signs1=self.signs1, signs2=self.signs2,
                                    rotation=self.rotation, norm_correction=self.norm_correction)
        return self._handle

    def _check(self, a, what):
        if a.shape[-1] != self.d:
            raise ValueError(f"{what}: last dimension must be {self.d}, got {a.shape[-1]}")

    def _launch_quantize(self, xd, idx, norms):
        """Device vectors [n, d] -> uint8 indices and float64 norms (tq_quantize_indices)."""
        L.check(L.lib().tq_quantize_indices(self.handle.h, L.ptr(xd), xd.shape[0], L.dtype_code(xd), L.ptr(idx), L.ptr(norms),
                                            None, L.stream_ptr()))

    def _launch_residual(self, xd, idx, norms, res):
        """xd minus the reconstruction of (uint8 idx, norms), float64."""
        L.check(L.lib().tq_dequantize_indices(self.handle.h, L.ptr(idx), L.ptr(norms), xd.shape[0], None, L.ptr(xd),
                                              L.dtype_code(xd), L.ptr(res), L.stream_ptr()))

    def _start_quantize(self, x2):
        """Host vectors [n, d] -> (block, indices, norms) on the device, nothing waited for after the upload."""
        tt = L.torch()
        xd = L.to_device(x2)
        n = xd.shape[0]
        buf, (idx, norms) = L.device_block(((n, self.d), tt.uint8), ((n,), tt.float64))
        self._launch_quantize(xd, idx, norms)
        return buf, idx, norms

    @staticmethod
    def _fetch(block):
        buf, idx, norms = block
        return L.fetch(buf, (idx, np.int64), (norms, np.float64))

    def quantize(self, x):
        """(indices int64, norms float64); 1-D input gives 1-D indices and a
        scalar norm (turboquant/polar_quant.py:56-85)."""
        x = np.asarray(x)
        single = x.ndim == 1
        x2 = x[None, :] if single else x
        self._check(x2, "quantize")
        idx_h, norms_h = self._fetch(self._start_quantize(x2))
        return (idx_h[0], norms_h[0]) if single else (idx_h, norms_h)

    def _launch_dequantize(self, idx, norms, out):
        """uint8 indices and norms on the device -> float64 reconstruction."""
        L.check(L.lib().tq_dequantize_indices(self.handle.h, L.ptr(idx), L.ptr(norms), idx.shape[0], L.ptr(out), None, L.TQ_F64,
                                              None, L.stream_ptr()))

    def dequantize(self, indices, norms):
        """Reconstruction, float64 (turboquant/polar_quant.py:87-119)."""
        indices = np.asarray(indices)
        single = indices.ndim == 1
        if single:
            indices = indices[None, :]
            norms = np.array([norms])
        self._check(indices, "dequantize")
        tt = L.torch()
        idx, nrm = L.upload_indices(indices, self.n_centroids, L.host_norms(norms, indices.shape[0]))
        buf, (out,) = L.device_block(((idx.shape[0], self.d), tt.float64))
        self._launch_dequantize(idx, nrm, out)
        out_h = L.fetch(buf, (out, np.float64))[0]
        return out_h[0] if single else out_h

    def _residual_of(self, x, indices, norms):
        """x - dequantize(indices, norms) for host arrays."""
        tt = L.torch()
        single = x.ndim == 1
        i2 = np.asarray(indices)[None, :] if single else np.asarray(indices)
        x2 = x[None, :] if single else x
        self._check(i2, "dequantize")
        self._check(x2, "quantize")
        xd = L.to_device(x2)
        idx, nrm = L.upload_indices(i2, self.n_centroids, L.host_norms(norms, i2.shape[0]))
        buf, (res,) = L.device_block((tuple(i2.shape), tt.float64))
        self._launch_residual(xd, idx, nrm, res)
        res_h = L.fetch(buf, (res, np.float64))[0]
        return res_h[0] if single else res_h

    def quantize_and_residual(self, x):
        """(indices, norms, x - dequantize(indices, norms)) (turboquant/polar_quant.py:121-132)."""
        x = np.asarray(x)
        single = x.ndim == 1
        x2 = x[None, :] if single else x
        if not L.unchanged(self, *METHODS[:1]):
            idx, norms = self.quantize(x)
            return idx, norms, self._residual_of(x, idx, norms)
        self._check(x2, "quantize")
        tt = L.torch()
        xd = L.to_device(x2)
        n = xd.shape[0]
        buf, (idx, norms, res) = L.device_block(((n, self.d), tt.uint8), ((n,), tt.float64), ((n, self.d), tt.float64))
        self._launch_quantize(xd, idx, norms)
        self._launch_residual(xd, idx, norms, res)
        idx_h, norms_h, res_h = L.fetch(buf, (idx, np.int64), (norms, np.float64), (res, np.float64))
        return (idx_h[0], norms_h[0], res_h[0]) if single else (idx_h, norms_h, res_h)


METHODS = (PolarQuant.quantize, PolarQuant.quantize_and_residual, PolarQuant.dequantize)    # for _lib.unchanged
