"""The NumPy classes' way between host arrays and the device: stages that stay on the device, staged copies of large
results, indices narrowed and checked, and the views of a compressed cache taken as the arrays they are.  Every result is
compared bit for bit with the plain way."""
import numpy as np
import pytest

import turboquant_plus_amd as tqa
from turboquant_plus_amd import _lib as L

pytestmark = pytest.mark.gpu


def test_turboquant_pipeline_equals_its_parts():
    """quantize / dequantize keep everything on the device between the stages: the same numbers as the classes' own
    methods one after the other, for one vector, a few (one copy) and enough for the staged copies."""
    tq = tqa.TurboQuant(96, 3, seed=9)
    for n in (1, 20, 9000):
        x = np.random.default_rng(n).standard_normal((n, 96))
        c = tq.quantize(x)
        idx, norms, res = tq.polar_quant.quantize_and_residual(x)
        signs, rnorms = tq.qjl.quantize(res)
        for got, want in ((c.mse_indices, idx), (c.vector_norms, norms), (c.qjl_signs, signs), (c.residual_norms, rnorms)):
            assert got.dtype == want.dtype and np.array_equal(got, want)
        assert np.array_equal(tq.dequantize(c, shrinkage=0.5), tq.polar_quant.dequantize(idx, norms) + tq.qjl.dequantize(signs, rnorms, 0.5))


@pytest.mark.parametrize("dtype,to", [("uint8", np.int64), ("int8", np.int8), ("float64", np.float64)])
@pytest.mark.parametrize("n", [1, 4095, L.ONE_COPY // 8 - 31, L.ONE_COPY + 1, 3_000_001, 2 * (L.STAGE // 8) + 17, 5_000_003])
def test_results_arrive_whole(dtype, to, n):
    tt = L.torch()
    dt = getattr(tt, dtype)
    buf, (a, b) = L.device_block(((n,), dt), ((3,), tt.float64))
    a.copy_(tt.randint(0, 100, (n,), device="cuda", generator=tt.Generator("cuda").manual_seed(n)))
    b.copy_(tt.tensor([1.5, -2.0, 3.0]))
    ha, hb = L.fetch(buf, (a, to), (b, np.float64))
    assert ha.dtype == to and np.array_equal(ha, a.cpu().numpy().astype(to)) and hb.tolist() == [1.5, -2.0, 3.0]


def test_indices_outside_the_codebook_are_refused():
    for n in (5, 700_000):
        i = np.random.default_rng(n).integers(0, 8, n)
        assert np.array_equal(L.narrow_indices(i, 8), i)
        for bad in (-1, 8, 1 << 40):
            j = i.copy()
            j[n // 2] = bad
            for dt in (np.int64, np.float64):
                with pytest.raises(ValueError, match="out of range"):
                    L.narrow_indices(j.astype(dt), 8)
    with pytest.raises(ValueError, match="norms"):
        tqa.PolarQuant(16, 2).dequantize(np.zeros((3, 16), dtype=np.int64), np.ones(2))


def test_views_of_one_cache_are_taken_together():
    """decompress() takes compress()'s (layer, head) views as the arrays they are; containers of other arrays give the same."""
    kv = tqa.KVCacheCompressor(32, k_bits=3, v_bits=2, seed=1)
    rng = np.random.default_rng(0)
    c = kv.compress(rng.standard_normal((2, 3, 7, 32)), rng.standard_normal((2, 3, 7, 32)))
    k, v = kv.decompress(c)
    for row in c.k_compressed:
        for e in row:
            e.mse_indices, e.qjl_signs, e.vector_norms = e.mse_indices.copy(), np.asfortranarray(e.qjl_signs), list(e.vector_norms)
    c.v_indices[1][2] = c.v_indices[1][2].astype(np.int32)
    k2, v2 = kv.decompress(c)
    assert np.array_equal(k, k2) and np.array_equal(v, v2)


def test_a_subclass_that_overrides_quantize():
    """The residual is that of the indices and norms which the subclass's quantize gives."""
    class Coarse(tqa.PolarQuant):
        def quantize(self, x):
            idx, norms = super().quantize(x)
            return idx | 1, norms
    own, other = tqa.PolarQuant(24, 3, seed=4), Coarse(24, 3, seed=4)
    for x in (np.random.default_rng(0).standard_normal((6, 24)), np.random.default_rng(1).standard_normal(24)):
        idx, norms, res = other.quantize_and_residual(x)
        assert np.array_equal(idx, own.quantize(x)[0] | 1) and np.array_equal(norms, own.quantize(x)[1])
        np.testing.assert_allclose(res, x - own.dequantize(idx, norms), atol=1e-13)
