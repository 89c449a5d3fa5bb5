"""The float64 dense products (rotation, reconstruction, projections) at the edges of their tiles.

Tolerance: a sum of d products in any order is off by at most d * 2^-53 * sum |m||x| <= d * 2^-53 * ||x|| for rows of an
orthogonal matrix, on each of the two sides compared; a few further roundings (norm, division, scale) add a constant."""
import numpy as np
import pytest

import tq_oracle as O
import turboquant_plus_amd as tqa
from turboquant_plus_amd import _lib as L

pytestmark = pytest.mark.gpu


def bound(d):
    return 2 * (d + 16) * 2.0 ** -53


# one vector and up to 16 (single tiles), one tile row more, several rows and a remainder; dimensions below, at and past a
# chunk of 16 values, a tile of 16 columns and the eight column blocks that are dealt to the XCDs; the last four go through
# the slices of their contraction in one wavefront: eight row groups a workgroup, the last ones past the end
@pytest.mark.parametrize("n,d", [(1, 1), (3, 2), (16, 16), (17, 15), (2, 17), (33, 31), (16, 130), (31, 33), (65, 64), (5, 250),
                                 (40, 257), (700, 129), (2100, 200), (4500, 272), (9001, 272),
                                 (40003, 100), (52001, 31), (6700, 600)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_dense_products_at_tile_edges(n, d, dtype):
    x = (np.random.default_rng(n * 1000 + d).standard_normal((n, d)) * np.logspace(-3, 3, n)[:, None]).astype(dtype)
    if n > 2:
        x[n // 2] = 0.0
    g, o = tqa.PolarQuant(d, 3, seed=7), O.PolarRef(d, 3, seed=7)
    idx, norms = g.quantize(x)
    y, no = o.rotated(x)
    np.testing.assert_allclose(norms, no, rtol=bound(d))
    mid = (o.centroids[:-1] + o.centroids[1:]) / 2
    want = np.searchsorted(mid, y.ravel(), side="left").reshape(y.shape)
    near = np.abs(y[..., None] - mid).min(axis=-1) <= bound(d)
    assert idx.dtype == np.int64 and np.array_equal(idx[~near], want[~near])
    i2, n2, res = g.quantize_and_residual(x)
    assert np.array_equal(i2, idx) and np.array_equal(n2, norms)
    xh = g.dequantize(idx, norms)
    tol = 4 * bound(d) * norms[:, None] + 1e-300
    assert np.all(np.abs(xh - o.dequantize(idx, norms)) <= tol)
    assert np.all(np.abs(res - (x.astype(np.float64) - xh)) <= tol)
    q, qo = tqa.QJL(d, seed=5), O.QJLRef(d, seed=5)
    s, rn = q.quantize(x)
    proj = qo.project(x.astype(np.float64))
    clear = np.abs(proj) > bound(d) * no[:, None]
    assert s.dtype == np.int8 and np.array_equal(s[clear], np.where(proj < 0, -1, 1)[clear])
    np.testing.assert_allclose(rn, no, rtol=bound(d))
    # signs have norm sqrt(d): the sums are that much larger than the result's scale * norm
    assert np.all(np.abs(q.dequantize(s, rn) - qo.dequantize(s, rn)) <= 4 * bound(d) * np.sqrt(d) * q.scale * rn[:, None] + 1e-300)


# the tile that a launch's workgroups are done first with: 1 x 1 past sixteen vectors (one column block a tile, seven or fewer
# and more than seven of them; several row groups a workgroup), 1 x 2, 2 x 2 and 2 x 3 with whole and cut tiles on both sides
@pytest.mark.parametrize("n,d", [(17, 16), (900, 23), (33, 250), (300, 300), (600, 128), (325, 601), (1200, 127), (400, 384), (513, 381),
                                 (1024, 384), (1023, 200), (2300, 128), (210, 1100), (137, 2048)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_dense_products_in_every_tile(n, d, dtype):
    test_dense_products_at_tile_edges(n, d, dtype)


@pytest.mark.parametrize("n,d", [(450, 64), (325, 601), (1000, 383), (256, 1100)])
def test_tiles_do_not_change_a_vector_s_results(n, d):
    """A vector's bits are those it has alone, in a single tile."""
    x = np.random.default_rng(n).standard_normal((n, d))
    tq = tqa.TurboQuant(d, 3)
    whole = tq.quantize(x)
    back = tq.dequantize(whole)
    for at in (0, 15, 16, n // 2, n - 1):
        part = tq.quantize(x[at:at + 1])
        for name in ("mse_indices", "vector_norms", "qjl_signs", "residual_norms"):
            assert np.array_equal(getattr(part, name), getattr(whole, name)[at:at + 1]), (name, at)
        assert np.array_equal(tq.dequantize(part), back[at:at + 1])


@pytest.mark.parametrize("bits", [1, 5, 8])
def test_level_search_at_every_width(bits):
    """The level of a value is the number of midpoints below it."""
    g = tqa.PolarQuant(64, bits, seed=3)
    x = np.random.default_rng(bits).standard_normal((300, 64))
    idx, norms = g.quantize(x)
    y, _ = O.PolarRef(64, bits, seed=3).rotated(x)
    mid = (g.centroids[:-1] + g.centroids[1:]) / 2
    near = np.abs(y[..., None] - mid).min(axis=-1) <= bound(64)
    assert np.array_equal(idx[~near], np.searchsorted(mid, y.ravel(), side="left").reshape(y.shape)[~near])
    w = tqa.PolarQuant(64, bits, seed=3, rotation="wht")
    assert np.array_equal(w.quantize(x)[0], O.PolarRef(64, bits, seed=3, rotation="wht").quantize(x)[0])


def quantize_indices(handle, x, rotated=None):
    """tq_quantize_indices on a device tensor: indices and norms as NumPy arrays (rotated: a device tensor or None)."""
    tt = L.torch()
    n, d = x.shape
    idx, norms = tt.empty((n, d), dtype=tt.uint8, device="cuda"), tt.empty(n, dtype=tt.float64, device="cuda")
    L.check(L.lib().tq_quantize_indices(handle.h, L.ptr(x), n, L.dtype_code(x), L.ptr(idx), L.ptr(norms), L.ptr(rotated), L.stream_ptr()))
    return idx.cpu().numpy(), norms.cpu().numpy()


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 6])
@pytest.mark.parametrize("rotation", ["dense", "wht"])
@pytest.mark.parametrize("order", ["shuffled", "with gaps"])
def test_codebooks_in_any_order(bits, rotation, order):
    """The code is the number of midpoints of neighbouring entries below the value, whatever their order."""
    d, rng = 96, np.random.default_rng(bits)
    cent = rng.uniform(-0.3, 0.3, 1 << bits)
    if order == "with gaps":
        cent[: 1 << (bits - 1)] = cent[0] * 100
    q = O.PolarRef(d, 3, seed=7, rotation=rotation)
    tables = dict(rotation=q.rotation) if rotation == "dense" else dict(signs1=q.s1, signs2=q.s2)
    x = rng.standard_normal((300, d))
    xd = L.torch().from_numpy(x).cuda()
    idx, _ = quantize_indices(L.Handle(d, bits, cent, **tables), xd)
    y, _ = q.rotated(x)
    mid = (cent[1:] + cent[:-1]) / 2
    clear = np.abs(y[..., None] - mid).min(axis=-1) > bound(2 * d)
    assert clear.mean() > 0.99 and np.array_equal(idx[clear], (mid < y[..., None]).sum(axis=-1)[clear])


def rotate(handle, x, out, transpose=0):
    """tq_rotate on device tensors."""
    L.check(L.lib().tq_rotate(handle.h, L.ptr(x), L.ptr(out), x.shape[0], L.dtype_code(x), L.dtype_code(out), transpose, L.stream_ptr()))
    return out


def rounding(dtype):
    """Half a unit in the last place, relative, and half of the smallest step of a type."""
    return {"float16": (2.0 ** -11, 2.0 ** -25), "float32": (2.0 ** -24, 2.0 ** -150), "float64": (2.0 ** -53, 0.0)}[dtype]


@pytest.mark.parametrize("n,d", [(1, 1), (1, 33), (16, 17), (17, 300), (65, 64), (1001, 130), (9, 1030), (5, 2100)])
@pytest.mark.parametrize("dtype", ["float16", "float32", "float64"])
def test_dense_results_in_the_memory_of_the_input(n, d, dtype):
    """Every column of a row needs the whole row: more than one column block reads what another one stores."""
    tt = L.torch()
    rng = np.random.default_rng(n + d)
    m = np.linalg.qr(rng.standard_normal((d, d)))[0]
    h = L.Handle(d, 3, np.sort(rng.uniform(-0.3, 0.3, 8)), rotation=m)
    x = tt.from_numpy(rng.standard_normal((n, d)).astype(dtype)).cuda()
    x64 = x.cpu().numpy().astype(np.float64)
    size = np.linalg.norm(x64, axis=1, keepdims=True)
    rel, step = rounding(dtype)
    for transpose, want in ((0, x64 @ m.T), (1, x64 @ m)):
        y = x.clone()
        rotate(h, y, y, transpose)
        assert np.all(np.abs(y.cpu().numpy().astype(np.float64) - want) <= (1 + 2.0 ** -20) * (rel * np.abs(want) + bound(d) * size) + step)
    if dtype == "float64":
        y = x.clone()
        idx, norms = quantize_indices(h, y, rotated=y)
        rotated = x64 @ m.T / size
        assert np.all(np.abs(y.cpu().numpy() - rotated) <= bound(d))
        np.testing.assert_allclose(norms, size[:, 0], rtol=bound(d))
        apart, idx_apart = tt.empty_like(x), quantize_indices(h, x, rotated=None)[0]
        quantize_indices(h, x, rotated=apart)
        assert np.all(np.abs(apart.cpu().numpy() - rotated) <= bound(d))
        assert (idx != idx_apart).mean() < 1e-3


@pytest.mark.parametrize("d", [5, 17, 40, 64, 100, 128, 200, 272, 384, 515])
def test_results_do_not_depend_on_the_batch(d):
    """A vector alone, in a batch of a tile row, of some and of many: the same bits, whatever launch each takes."""
    n = 70_003 if d < 300 else 9_001          # unsplit products
    x = np.random.default_rng(d).standard_normal((n, d))
    tq = tqa.TurboQuant(d, 3)
    g = tq.polar_quant
    whole = tq.quantize(x)
    residual = g.quantize_and_residual(x[:3000])[2]
    back = tq.dequantize(whole)
    for size in (1, 16, 17, 40, 600, 3000):
        for at in (0, n - size):
            part = tq.quantize(x[at:at + size])
            for name in ("mse_indices", "vector_norms", "qjl_signs", "residual_norms"):
                assert np.array_equal(getattr(part, name), getattr(whole, name)[at:at + size]), (name, size)
            assert np.array_equal(tq.dequantize(part), back[at:at + size])
        assert np.array_equal(g.quantize_and_residual(x[:size])[2], residual[:size])


@pytest.mark.parametrize("n", [3, 40])
@pytest.mark.parametrize("rotation", ["dense", "wht"])
def test_indices_past_the_codebook(rotation, n):
    """They stand for its last entry, in both modes."""
    tt = L.torch()
    d, q = 48, O.PolarRef(48, 3, seed=7, rotation=rotation)
    tables = dict(rotation=q.rotation) if rotation == "dense" else dict(signs1=q.s1, signs2=q.s2)
    h = L.Handle(d, 3, q.centroids, **tables)
    idx = np.random.default_rng(n).integers(0, 256, (n, d)).astype(np.uint8)
    norms, out = np.linspace(0.5, 2, n), tt.empty((n, d), dtype=tt.float64, device="cuda")
    idx_d, norms_d = tt.from_numpy(idx).cuda(), tt.from_numpy(norms).cuda()
    L.check(L.lib().tq_dequantize_indices(h.h, L.ptr(idx_d), L.ptr(norms_d), n, L.ptr(out), None, L.TQ_F64, None, L.stream_ptr()))
    np.testing.assert_allclose(out.cpu().numpy(), q.dequantize(np.minimum(idx, 7), norms), atol=4 * bound(d) * 2)


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("rotation", ["dense", "wht"])
def test_values_on_a_midpoint_and_nan(bits, rotation):
    """A value equal to a midpoint takes the level below it, NaN level 0.  Every step is exact: midpoints are multiples of
    1/8 (or of a finer power of two), rows have norm 1 and entries 0, +-1/2, +-1/4 or +-1/8, the rotation is the identity or a
    butterfly that gives them back."""
    d, rng = 64, np.random.default_rng(bits)
    rows = np.zeros((96, d))
    for r in range(96):
        count = (4, 16, 64)[r % 3]
        rows[r, rng.permutation(d)[:count]] = rng.choice([-1.0, 1.0], count) / np.sqrt(count)
    cent = (np.arange(1 << bits) + 0.5) / (1 << (bits - 1)) - 1.0
    mid = (cent[:-1] + cent[1:]) / 2
    assert bits == 1 or np.isin(rows, mid).any()
    if rotation == "dense":
        h, x = L.Handle(d, bits, cent, rotation=np.eye(d)), rows.copy()
    else:
        h, x = L.Handle(d, bits, cent, signs1=np.ones(d), signs2=np.ones(d)), O.rotate_fast(rows, np.ones(d), np.ones(d), d)
    x[5, 7] = np.nan
    tt = L.torch()
    for n in (1, 40, 96):
        idx, norms = quantize_indices(h, tt.from_numpy(x[:n]).cuda())
        want = np.searchsorted(mid, rows[:n].ravel(), side="left").reshape(n, d)
        if n > 5:
            want[5] = 0
            assert np.isnan(norms[5])
        assert np.array_equal(idx, want) and np.array_equal(np.delete(norms, 5) if n > 5 else norms, np.ones(n - (n > 5)))


@pytest.mark.parametrize("n,d", [(3, 40), (100, 130), (60_000, 33)])
@pytest.mark.parametrize("dtype", ["float16", "float32", "float64"])
@pytest.mark.parametrize("out_dtype", ["float16", "float32", "float64"])
def test_dense_rotation(n, d, dtype, out_dtype):
    """tq_rotate on a dense handle, forward and transposed, every pair of types in each of the launches."""
    tt = L.torch()
    rng = np.random.default_rng(n + d)
    m = np.linalg.qr(rng.standard_normal((d, d)))[0]
    h = L.Handle(d, 2, np.linspace(-0.3, 0.3, 4), rotation=m)
    x = tt.from_numpy(rng.standard_normal((n, d)).astype(dtype)).cuda()
    x64 = x.cpu().numpy().astype(np.float64)
    size = np.linalg.norm(x64, axis=1, keepdims=True)
    rel, step = rounding(out_dtype)
    for transpose, want in ((0, x64 @ m.T), (1, x64 @ m)):
        y = rotate(h, x, tt.empty((n, d), dtype=getattr(tt, out_dtype), device="cuda"), transpose)
        # fp16 results are rounded to fp32 on the way
        assert np.all(np.abs(y.cpu().numpy().astype(np.float64) - want) <= (1 + 2.0 ** -10) * (rel * np.abs(want) + bound(d) * size) + step)


@pytest.mark.parametrize("n", [8, 40, 300])
@pytest.mark.parametrize("rotation", ["dense", "wht"])
def test_rows_whose_norm_is_past_the_range(rotation, n):
    """Finite entries over an infinite norm are zeros (their sums may overflow first); an infinite entry makes NaN."""
    d, rng = 100, np.random.default_rng(n)
    q = O.PolarRef(d, 3, seed=7, rotation=rotation)
    tables = dict(rotation=q.rotation) if rotation == "dense" else dict(signs1=q.s1, signs2=q.s2)
    h = L.Handle(d, 3, q.centroids, **tables)
    x = rng.standard_normal((n, d))
    x[0] = rng.choice([-1.0, 1.0], d) * 1.7e308
    x[1] = 1.7e308
    x[2] *= 1e200
    x[3, 5] = -np.inf
    tt = L.torch()
    rotated = tt.empty((n, d), dtype=tt.float64, device="cuda")
    idx, norms = quantize_indices(h, tt.from_numpy(x).cuda(), rotated=rotated)
    zero = int((((q.centroids[1:] + q.centroids[:-1]) / 2) < 0.0).sum())
    y = rotated.cpu().numpy()
    assert (idx[:3] == zero).all() and (y[:3] == 0.0).all() and np.isinf(norms[:4]).all()
    assert (idx[3] == 0).all() and np.isnan(y[3]).all()
    want, wn = q.quantize(x[4:])
    assert (idx[4:] != want).mean() < 1e-3 and np.allclose(norms[4:], wn, rtol=1e-13)
