"""Host-array handling of the NumPy classes that needs no GPU."""
import os
import subprocess
import sys

import numpy as np
import pytest

from turboquant_plus_amd import _lib as L
from turboquant_plus_amd.kv_cache import KVCacheCompressor, _joined
from turboquant_plus_amd.polar_quant import PolarQuant
from turboquant_plus_amd.qjl import QJL
from turboquant_plus_amd.turboquant import CompressedVector, TurboQuant

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("t", [0, 1, 4])
def test_one_token_pieces_of_a_token_major_container(t):
    """A piece of one token is contiguous whatever the stride of its token axis: heads of one token in containers
    [tokens, heads, d] and [tokens, heads] are neighbours in memory whose stride along tokens is not theirs to use."""
    x = np.arange(60).reshape(5, 3, 4)
    joined = _joined([x[t:t + 1, h] for h in range(3)])
    assert joined.flags.c_contiguous and np.array_equal(joined, x[t])
    norms = np.arange(15.0).reshape(5, 3)
    assert np.array_equal(_joined([norms[t:t + 1, h] for h in range(3)]), norms[t])
    one = np.arange(4.0).reshape(1, 4)
    assert np.array_equal(_joined([one[:, h] for h in range(4)]), one[0])


def test_joined_equals_concatenate():
    """Pieces of one array, neighbours or not, in any order and of any axis order."""
    x = np.random.default_rng(0).standard_normal((2, 3, 5, 4))
    for a in (x, x.transpose(1, 0, 2, 3), x.transpose(2, 1, 0, 3), x[::-1], x[:, :, ::2], x[..., ::-1], x[:, :, :1], np.asfortranarray(x)):
        for pieces in ([a[i, j] for i in range(a.shape[0]) for j in range(a.shape[1])], [a[i, 0] for i in range(a.shape[0])],
                       [a[0, 0], a[0, 0]], [a[0, 0]], [a[0, 0], a[0, 1].astype(np.float32)]):
            assert np.array_equal(_joined(pieces), np.concatenate(pieces, axis=0))


def test_scalar_norms_join():
    """Containers of one token may hold a plain number per (layer, head)."""
    for scalars in ([np.float64(2.5), 3, np.array(4.0)], list(np.arange(3.0)[:, None].T.reshape(3))):
        assert np.array_equal(_joined(scalars), np.asarray(scalars, dtype=np.float64))
    z = np.arange(3.0)
    assert np.array_equal(_joined([z[i:i + 1].reshape(()) for i in range(3)]), z)


@pytest.mark.parametrize("when", ["after a fork", "at exit", "in a thread that outlives the main one"])
def test_copy_threads_that_are_not_there(when):
    """A call with large host arrays begins and ends where the copy threads are gone: in a forked child, and once the interpreter
    ends."""
    code = """
import atexit, os, sys, threading, time
import numpy as np
from turboquant_plus_amd import _lib as L
i = np.random.default_rng(0).integers(0, 8, 700_000)
def narrow():
    with L.helpers(L.SHARED + 1), L.helpers(L.SHARED + 1):
        assert np.array_equal(L.narrow_indices(i, 8), i)
    assert getattr(L._helping, "board", None) is None
    print("done", flush=True)
narrow()
together = threading.Barrier(L.COPY_THREADS)
for w in [L._copy_pool().submit(together.wait) for _ in range(L.COPY_THREADS)]:   # every thread has started
    w.result()
"""
    code += {"after a fork": "pid = os.fork()\nif pid == 0:\n    narrow()\n    os._exit(0)\n"
                             "end = time.time() + 30\nwhile time.time() < end and os.waitpid(pid, os.WNOHANG)[0] == 0:\n    time.sleep(0.05)\n"
                             "if time.time() >= end:\n    os.kill(pid, 9)\n    os.waitpid(pid, 0)\n",
             "at exit": "atexit.register(narrow)\n",
             "in a thread that outlives the main one": "def late():\n    threading.main_thread().join()\n    time.sleep(0.3)\n    narrow()\n"
                                                       "threading.Thread(target=late).start()\n"}[when]
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.count("done") == 2, out.stdout + out.stderr


def test_more_norms_than_vectors():
    """Norms past the last vector are not used; too few are refused."""
    assert L.host_norms(np.arange(5.0), 3).tolist() == [0.0, 1.0, 2.0]
    assert L.host_norms([[1, 2], [3, 4]], 4).tolist() == [1.0, 2.0, 3.0, 4.0]
    assert L.host_norms(np.arange(12.0).reshape(3, 4)[:, ::2], 5).flags.c_contiguous
    with pytest.raises(ValueError, match="norms"):
        L.host_norms(np.ones(2), 3)


class _Part:
    """A quantiser stage with the public methods only."""

    def __init__(self, d):
        self.d = d

    def dequantize(self, codes, norms, shrinkage=1.0):
        return np.asarray(codes) * (np.asarray(norms)[..., None] * shrinkage)


@pytest.mark.parametrize("idx,signs", [((5, 8), (1, 8)), ((5, 8), (8,)), ((1, 8), (5, 8)), ((8,), (5, 8))])
def test_signs_that_broadcast_against_indices(idx, signs):
    """TurboQuant.dequantize is the sum of its two stages' results, also where their shapes broadcast."""
    tq = TurboQuant(8, 3)
    tq.polar_quant, tq.qjl = _Part(8), _Part(8)
    rng = np.random.default_rng(1)
    i, s = rng.integers(0, 4, idx), rng.choice([-1, 1], signs).astype(np.int8)
    n, rn = rng.random(idx[:-1]), rng.random(signs[:-1])
    got = tq.dequantize(CompressedVector(i, n, s, rn, 3), shrinkage=0.5)
    assert np.array_equal(got, i * n[..., None] + s * rn[..., None] * 0.5)


class _Recorder:
    """The public methods of every stage, without a GPU."""

    def __init__(self, d):
        self.d = d

    def quantize(self, x):
        return np.sign(x).astype(np.int64), np.abs(x).sum(axis=-1)

    def quantize_and_residual(self, x):
        return (*self.quantize(x), x * 0.25)


def test_replaced_stages_are_asked_through_their_public_methods():
    tq = TurboQuant(8, 3)
    tq.polar_quant, tq.qjl = _Recorder(8), _Recorder(8)
    x = np.random.default_rng(2).standard_normal((5, 8))
    for rows in (x, x[0]):
        c = tq.quantize(rows)
        assert np.array_equal(c.mse_indices, np.sign(rows)) and np.array_equal(c.residual_norms, np.abs(rows * 0.25).sum(axis=-1))
        assert c.bit_width == 3
    kv = KVCacheCompressor(8)
    kv.k_quantizer, kv.v_quantizer.polar_quant = tq, _Recorder(8)
    k = np.random.default_rng(3).standard_normal((2, 3, 5, 8))
    c = kv.compress(k, -k)
    assert np.array_equal(c.k_compressed[1][2].mse_indices, np.sign(k[1, 2]))
    assert np.array_equal(c.v_indices[0][1], np.sign(-k[0, 1])) and np.array_equal(c.v_norms[1][0], np.abs(k[1, 0]).sum(axis=-1))


def test_overridden_methods_are_called(monkeypatch):
    """In a subclass, on an object, on the class."""
    class Polar(PolarQuant):
        def quantize(self, x):
            return np.full(np.shape(x), 7), np.zeros(np.shape(x)[:-1])

        def _residual_of(self, x, idx, norms):      # what follows on the device
            return idx * 2.0
    idx, _, res = Polar(8, 3).quantize_and_residual(np.ones((2, 8)))
    assert (idx == 7).all() and (res == 14).all()
    tq = TurboQuant(8, 3)
    tq.polar_quant.quantize_and_residual = lambda x: (1, 2, 3)
    monkeypatch.setattr(QJL, "quantize", lambda self, r: (r, r))
    c = tq.quantize(np.ones((2, 8)))
    assert (c.mse_indices, c.vector_norms, c.qjl_signs) == (1, 2, 3)
    tq = TurboQuant(8, 3)
    tq.polar_quant.dequantize = tq.qjl.dequantize = lambda *a, **k: 1.0
    z = np.zeros((2, 8), np.int64)
    assert tq.dequantize(CompressedVector(z, z[:, 0], z, z[:, 0], 3)) == 2.0
    kv = KVCacheCompressor(8)
    kv.k_quantizer.quantize = lambda x: CompressedVector(x, x[:, 0], x, x[:, 1], 3)
    kv.v_quantizer.quantize = lambda x: (x, x[:, 2])
    k = np.random.default_rng(3).standard_normal((2, 3, 5, 8))
    c = kv.compress(k, k)
    assert np.array_equal(c.k_compressed[1][1].residual_norms, k[1, 1, :, 1]) and np.array_equal(c.v_norms[0][2], k[0, 2, :, 2])
