"""TurboQuant = PolarQuant at b-1 bits + 1-bit QJL on the residual, and the
MSE-only variant, with the reference's interface (turboquant/turboquant.py:33-171)."""
from __future__ import annotations

from dataclasses import dataclass

import numpy as np

from . import _lib as L
from . import polar_quant, qjl
from .polar_quant import PolarQuant
from .qjl import QJL


@dataclass
class CompressedVector:
    """turboquant/turboquant.py:33-40."""
    mse_indices: np.ndarray     # (d,) or (batch, d), (b-1)-bit codebook indices
    vector_norms: np.ndarray    # scalar or (batch,), ||x||
    qjl_signs: np.ndarray       # (d,) or (batch, d), int8 {+1,-1}
    residual_norms: np.ndarray  # scalar or (batch,), ||x - x_mse||
    bit_width: int              # total bits per coordinate


class TurboQuant:
    def __init__(self, d: int, bit_width: int, seed: int = 42, norm_correction: bool = True, *,
                 rotation: str = "dense", projection: str = "orthogonal"):
        if bit_width < 2:
            raise ValueError("TurboQuant requires bit_width >= 2 (1 bit PolarQuant + 1 bit QJL). "
                             "For 1-bit, use QJL directly.")
        self.d = d
        self.bit_width = bit_width
        self.polar_quant = PolarQuant(d, bit_width=bit_width - 1, seed=seed, norm_correction=norm_correction,
                                      rotation=rotation)
        self.qjl = QJL(d, seed=seed + 1000, projection=projection)  # turboquant/turboquant.py:77

    # Both directions stay on the device between the stages: indices, norms and the residual are handed over there, and
    # only what the caller gets crosses to the host.
    def _on_device(self):
        return L.unchanged(self.polar_quant, *polar_quant.METHODS) and L.unchanged(self.qjl, *qjl.METHODS)

    def _launch_quantize(self, xd):
        """Device vectors [n, d] -> (block, indices uint8, norms, signs, residual norms) on the device."""
        tt = L.torch()
        n = xd.shape[0]
        buf, (idx, norms, signs, rnorms) = L.device_block(((n, self.d), tt.uint8), ((n,), tt.float64), ((n, self.d), tt.int8),
                                                          ((n,), tt.float64))
        res = tt.empty((n, self.d), dtype=tt.float64, device=xd.device)
        self.polar_quant._launch_quantize(xd, idx, norms)
        self.polar_quant._launch_residual(xd, idx, norms, res)
        self.qjl._launch_quantize(res, signs, rnorms)
        return buf, idx, norms, signs, rnorms

    @staticmethod
    def _fetch(block):
        buf, idx, norms, signs, rnorms = block
        return L.fetch(buf, (idx, np.int64), (norms, np.float64), (signs, np.int8), (rnorms, np.float64))

    def quantize(self, x) -> CompressedVector:
        x = np.asarray(x)
        single = x.ndim == 1
        x2 = x[None, :] if single else x
        if not self._on_device():
            idx, norms, residual = self.polar_quant.quantize_and_residual(x)
            signs, rnorms = self.qjl.quantize(residual)
        else:
            self.polar_quant._check(x2, "quantize")
            with L.helpers(8 * x2.size):
                idx, norms, signs, rnorms = self._fetch(self._launch_quantize(L.to_device(x2)))
            if single:
                idx, norms, signs, rnorms = idx[0], norms[0], signs[0], rnorms[0]
        return CompressedVector(mse_indices=idx, vector_norms=norms, qjl_signs=signs, residual_norms=rnorms,
                                bit_width=self.bit_width)

    def dequantize(self, compressed: CompressedVector, shrinkage: float = 1.0):
        idx, signs = np.asarray(compressed.mse_indices), np.asarray(compressed.qjl_signs)
        norms, rnorms = compressed.vector_norms, compressed.residual_norms
        if signs.shape != idx.shape or not self._on_device():    # shapes may broadcast: the sum of two results
            return self.polar_quant.dequantize(idx, norms) + self.qjl.dequantize(signs, rnorms, shrinkage=shrinkage)
        single = idx.ndim == 1
        if single:
            idx, signs, norms, rnorms = idx[None, :], signs[None, :], np.array([norms]), np.array([rnorms])
        self.polar_quant._check(idx, "dequantize")
        n = idx.shape[0]
        tt = L.torch()
        with L.helpers(8 * idx.size):
            idx_d, norms_d, signs_d, rnorms_d = L.upload_indices(idx, self.polar_quant.n_centroids, L.host_norms(norms, n),
                                                                 np.ascontiguousarray(signs, dtype=np.int8), L.host_norms(rnorms, n))
            buf, (out,) = L.device_block(((n, self.d), tt.float64))
            self.polar_quant._launch_dequantize(idx_d, norms_d, out)
            self.qjl._launch_dequantize(signs_d, rnorms_d, shrinkage, out, add=True)
            out_h = L.fetch(buf, (out, np.float64))[0]
        return out_h[0] if single else out_h

    def compressed_size_bits(self, n_vectors: int) -> int:
        """b bits per coordinate plus one 32-bit norm per vector (turboquant/turboquant.py:126-136)."""
        return n_vectors * (self.d * self.bit_width + 32)

    def compression_ratio(self, original_bits_per_value: int = 16) -> float:
        return (self.d * original_bits_per_value) / (self.d * self.bit_width + 32)


class TurboQuantMSE:
    """PolarQuant at the full bit width, no QJL stage (turboquant/turboquant.py:152-171)."""

    def __init__(self, d: int, bit_width: int, seed: int = 42, norm_correction: bool = True, *,
                 rotation: str = "dense"):
        self.d = d
        self.bit_width = bit_width
        self.polar_quant = PolarQuant(d, bit_width=bit_width, seed=seed, norm_correction=norm_correction,
                                      rotation=rotation)

    def quantize(self, x):
        return self.polar_quant.quantize(x)

    def dequantize(self, indices, norms):
        return self.polar_quant.dequantize(indices, norms)


METHODS = (TurboQuant.quantize, TurboQuant.dequantize)    # for _lib.unchanged
MSE_METHODS = (TurboQuantMSE.quantize, TurboQuantMSE.dequantize)
