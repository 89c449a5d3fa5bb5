"""KV-cache compressor with the reference's interface (turboquant/kv_cache.py:30-188).

One K quantiser (TurboQuant, seed) and one V quantiser (TurboQuantMSE,
seed + 500) serve every layer and head, so the reference's layers x heads loop
collapses into one kernel launch over all L*H*S vectors; the per-(layer, head)
containers are views of that result.
"""
from __future__ import annotations

from dataclasses import dataclass, field

import numpy as np

from . import _lib as lib
from . import polar_quant, turboquant
from .turboquant import CompressedVector, TurboQuant, TurboQuantMSE


@dataclass
class CompressedKVCache:
    """turboquant/kv_cache.py:30-44."""
    k_compressed: list = field(default_factory=list)   # [layer][head] CompressedVector over seq
    v_indices: list = field(default_factory=list)      # [layer][head] (seq, head_dim)
    v_norms: list = field(default_factory=list)        # [layer][head] (seq,)
    num_layers: int = 0
    num_heads: int = 0
    seq_len: int = 0
    head_dim: int = 0
    k_bit_width: int = 0
    v_bit_width: int = 0


def _joined(pieces):
    """The (layer, head) arrays one after another.  compress() hands out views that follow each other in one array: pieces
    of one base whose memory is adjacent are taken as the stretch they are, others are copied together.  The stretch gets
    the strides of its shape: a piece is contiguous whatever stride its axes of one entry have, and those strides (of a
    token-major container, say) lead elsewhere."""
    pieces = [np.atleast_1d(np.asarray(p)) for p in pieces]     # the norm of one token may be a plain number
    first = pieces[0]
    at = first.__array_interface__["data"][0]
    for p in pieces:
        if (first.base is None or p.base is not first.base or p.dtype != first.dtype or p.shape != first.shape
                or not p.flags.c_contiguous or p.__array_interface__["data"][0] != at):
            return np.concatenate(pieces, axis=0)
        at += p.nbytes
    shape = (len(pieces) * first.shape[0],) + first.shape[1:]
    strides = [first.itemsize]
    for n in shape[:0:-1]:
        strides.insert(0, n * strides[0])
    return np.lib.stride_tricks.as_strided(first, shape, strides)


class KVCacheCompressor:
    def __init__(self, head_dim: int, k_bits: int = 3, v_bits: int = 3, seed: int = 42,
                 norm_correction: bool = True):
        self.head_dim = head_dim
        self.k_bits = k_bits
        self.v_bits = v_bits
        self.k_quantizer = TurboQuant(head_dim, bit_width=k_bits, seed=seed, norm_correction=norm_correction)
        self.v_quantizer = TurboQuantMSE(head_dim, bit_width=v_bits, seed=seed + 500,
                                         norm_correction=norm_correction)

    def _on_device(self):
        k, v = self.k_quantizer, self.v_quantizer
        return (lib.unchanged(k, *turboquant.METHODS) and k._on_device() and lib.unchanged(v, *turboquant.MSE_METHODS)
                and lib.unchanged(v.polar_quant, *polar_quant.METHODS))

    def compress(self, k_cache: np.ndarray, v_cache: np.ndarray) -> CompressedKVCache:
        L, H, S, D = k_cache.shape
        assert D == self.head_dim
        assert v_cache.shape == k_cache.shape
        out = CompressedKVCache(num_layers=L, num_heads=H, seq_len=S, head_dim=D,
                                k_bit_width=self.k_bits, v_bit_width=self.v_bits)
        k_rows, v_rows = np.asarray(k_cache).reshape(L * H * S, D), np.asarray(v_cache).reshape(L * H * S, D)
        if self._on_device():   # both tensors are on their way before the first results are waited for
            kq, vq = self.k_quantizer, self.v_quantizer.polar_quant
            with lib.helpers(8 * k_rows.size):     # results of 8 bytes per value
                k_block = kq._launch_quantize(lib.to_device(k_rows))
                v_block = vq._start_quantize(v_rows)
                k_idx, k_nrm, k_sgn, k_rn = kq._fetch(k_block)
                vi, vn = vq._fetch(v_block)
        else:
            kc = self.k_quantizer.quantize(k_rows)
            k_idx, k_nrm, k_sgn, k_rn = kc.mse_indices, kc.vector_norms, kc.qjl_signs, kc.residual_norms
            vi, vn = self.v_quantizer.quantize(v_rows)
        k_idx, k_sgn, vi = (a.reshape(L, H, S, D) for a in (k_idx, k_sgn, vi))
        k_nrm, k_rn, vn = (a.reshape(L, H, S) for a in (k_nrm, k_rn, vn))
        for l in range(L):
            out.k_compressed.append([CompressedVector(k_idx[l, h], k_nrm[l, h], k_sgn[l, h], k_rn[l, h], self.k_bits)
                                     for h in range(H)])
            out.v_indices.append([vi[l, h] for h in range(H)])
            out.v_norms.append([vn[l, h] for h in range(H)])
        return out

    def decompress(self, compressed: CompressedKVCache):
        L, H, S, D = compressed.num_layers, compressed.num_heads, compressed.seq_len, compressed.head_dim
        flat = [compressed.k_compressed[l][h] for l in range(L) for h in range(H)]
        if not flat or S == 0:
            z = np.zeros((L, H, S, D))
            return z, z.copy()
        kc = CompressedVector(_joined([c.mse_indices for c in flat]), _joined([c.vector_norms for c in flat]),
                              _joined([c.qjl_signs for c in flat]), _joined([c.residual_norms for c in flat]), self.k_bits)
        vi = _joined([compressed.v_indices[l][h] for l in range(L) for h in range(H)])
        vn = _joined([compressed.v_norms[l][h] for l in range(L) for h in range(H)])
        with lib.helpers(8 * L * H * S * D if self._on_device() else 0):
            k = self.k_quantizer.dequantize(kc).reshape(L, H, S, D)
            v = self.v_quantizer.dequantize(vi, vn).reshape(L, H, S, D)
        return k, v

    def memory_stats(self, seq_len: int, num_layers: int, num_heads: int) -> dict:
        """turboquant/kv_cache.py:167-188: K counts b bits + a 32-bit norm, V counts b bits."""
        n = num_layers * num_heads * seq_len
        original = n * self.head_dim * 2
        compressed = (n * (self.head_dim * self.k_bits + 32) + n * self.head_dim * self.v_bits) / 8
        return {
            "original_mb": original / 1024 / 1024,
            "compressed_mb": compressed / 1024 / 1024,
            "compression_ratio": original / compressed,
            "k_bits_per_value": self.k_bits,
            "v_bits_per_value": self.v_bits,
        }
