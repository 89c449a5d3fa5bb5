"""Appends whose first and last token fall on, before and behind the edges of the append kernels' units: the 16-token
groups of a V tile (a thread per row and group), the four tokens of a 16-lane row, the 128-token block.  The oracle is the
store of the whole sequence with the same arithmetic (float64 rows for the turbo formats), byte for byte."""
import ctypes as C

import numpy as np
import pytest

import tq_oracle as O
import turboquant_plus_amd as tqa
from turboquant_plus_amd import _lib as L
from test_gpu_turbo import check_codes, np_

pytestmark = pytest.mark.gpu
SPANS = [(0, 1), (0, 16), (0, 127), (1, 15), (15, 1), (15, 2), (16, 16), (17, 30), (31, 33), (47, 81), (63, 1), (63, 66), (64, 63),
         (79, 49), (112, 16), (113, 15), (126, 3), (127, 1), (127, 130), (130, 256)]
N_SEQS, CAPACITY, D = 2, 512, 128


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("kind", ["k", "v"])
def test_turbo_rows(bits, kind):
    codec = tqa.TurboCodec(bits, seed=3)
    x = np.random.default_rng(bits).standard_normal((N_SEQS, 400, D))
    x[0, 20] = 0
    for pos, n_new in SPANS:
        cache = L.torch().full((tqa.packed_bytes(bits, N_SEQS, CAPACITY),), 0xA5, dtype=L.torch().uint8, device="cuda")
        if pos:
            codec.append(x[:, 200:200 + pos], cache, 0, CAPACITY, kind=kind)
        codec.append(x[:, :n_new], cache, pos, CAPACITY, kind=kind)
        want = np_(codec.store(np.concatenate([x[:, 200:200 + pos], x[:, :n_new]], axis=1), kind=kind)).reshape(N_SEQS, -1, O.block_bytes(bits))
        got = np_(cache).reshape(N_SEQS, -1, O.block_bytes(bits))
        assert np.array_equal(got[:, :want.shape[1]], want), (pos, n_new)
        assert (got[:, want.shape[1]:] == 0xA5).all(), (pos, n_new)


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("kind", ["k", "v"])
@pytest.mark.parametrize("dtype,on_device", [("float16", False), ("float16", True), ("float32", False)])
def test_turbo_rows_on_the_matrix_cores(bits, kind, dtype, on_device):
    """float16 and float32 rows go through the matrix cores in units of 16 tokens.  Whatever tokens stay before a span (all-zero rows among
    both), the bytes are those of one append of all of them, whose codes and norms agree with the oracle, and nothing
    outside the touched blocks is written."""
    tt = L.torch()
    codec = tqa.TurboCodec(bits, seed=3)
    x = tt.randn((N_SEQS, 400, D), generator=tt.Generator("cuda").manual_seed(bits), device="cuda")
    if dtype == "float32":      # norms over seven decades
        x *= 10 ** (tt.rand((N_SEQS, 400, 1), generator=tt.Generator("cuda").manual_seed(5), device="cuda") * 7 - 4)
    x = x.to(getattr(tt, dtype))
    x[0, 20] = x[1, 203] = 0
    for pos, n_new in SPANS:
        rows = tt.cat([x[:, 200:200 + pos], x[:, :n_new]], dim=1)
        want, got = (tt.full((tqa.packed_bytes(bits, N_SEQS, CAPACITY),), 0xA5, dtype=tt.uint8, device="cuda") for _ in range(2))
        codec.append(rows, want, 0, CAPACITY, kind=kind)
        if pos:
            codec.append(x[:, 200:200 + pos], got, 0, CAPACITY, kind=kind)
        codec.append(x[:, :n_new], got, tt.tensor([pos], device="cuda") if on_device else pos, CAPACITY, kind=kind)
        assert tt.equal(got, want), (pos, n_new)
        blocks = -(-(pos + n_new) // 128)
        assert bool((got.view(N_SEQS, -1, O.block_bytes(bits))[:, blocks:] == 0xA5).all()), (pos, n_new)
        idx, g = (np_(a)[:, :pos + n_new] for a in codec.unpack_codes(got, N_SEQS, CAPACITY, kind=kind))
        check_codes(codec, np_(rows).reshape(-1, D), idx.reshape(-1, D), g.reshape(-1))


@pytest.mark.parametrize("kind", ["k", "v"])
@pytest.mark.parametrize("dtype", ["float16", "float32", "float64"])
@pytest.mark.parametrize("shift", [0, 1])
def test_q8_0_rows(kind, dtype, shift):
    """shift: rows that start one value behind a 16-byte boundary."""
    tt = L.torch()
    row = 128 * 136
    flat = tt.randn(N_SEQS * 400 * D, generator=tt.Generator("cuda").manual_seed(5), device="cuda", dtype=tt.float32).to(getattr(tt, dtype))
    x = flat.reshape(N_SEQS, 400, D)
    x[0, 20] = 0
    x[1, 3, 40] = float("inf")

    def rows(lo, n):
        buf = tt.empty(N_SEQS * n * D + 8, dtype=x.dtype, device="cuda")
        out = buf[shift:shift + N_SEQS * n * D].view(N_SEQS, n, D)
        out.copy_(x[:, lo:lo + n])
        assert (out.data_ptr() % 16 != 0) == bool(shift and x.element_size() * shift % 16)
        return out
    for pos, n_new in SPANS:
        cache = tt.full((N_SEQS * CAPACITY // 128 * row,), 0xA5, dtype=tt.uint8, device="cuda")
        if pos:
            tqa.q8_0_append(rows(200, pos), cache, 0, CAPACITY, kind=kind)
        tqa.q8_0_append(rows(0, n_new), cache, pos, CAPACITY, kind=kind)
        want = np_(tqa.q8_0_store(tt.cat([x[:, 200:200 + pos], x[:, :n_new]], dim=1), kind=kind)[0]).reshape(N_SEQS, -1, row)
        got = np_(cache).reshape(N_SEQS, -1, row)
        assert np.array_equal(got[:, :want.shape[1]], want), (pos, n_new)
        assert (got[:, want.shape[1]:] == 0xA5).all(), (pos, n_new)


@pytest.mark.parametrize("fmt", [("q8_0", "q8_0"), ("q8_0", "turbo2"), ("q8_0", "turbo3"), ("q8_0", "turbo4"), ("turbo2", "q8_0"),
                                 ("turbo3", "q8_0"), ("turbo4", "q8_0")])
@pytest.mark.parametrize("dtypes", [("float16", "float16"), ("float32", "float32"), ("float64", "float64"), ("float16", "float32")])
def test_layer_with_8_bit_rows(fmt, dtypes):
    """K and V of a step in one launch write the bytes of an append per side, with the position on the host and on the
    device; rows of different types keep taking two calls, and a position that does not fit writes nothing."""
    tt = L.torch()
    layer = tqa.LayerKV(tqa.LayerFormat(*fmt))
    gen = tt.Generator("cuda").manual_seed(1)
    k = tt.randn((N_SEQS, 400, D), generator=gen, device="cuda").to(getattr(tt, dtypes[0]))
    v = tt.randn((N_SEQS, 400, D), generator=gen, device="cuda").to(getattr(tt, dtypes[1]))
    one, two, dev = (layer.new_cache(N_SEQS, CAPACITY) for _ in range(3))
    over = tt.zeros(1, dtype=tt.int32, device="cuda")
    pos = 0
    for n_new in (1, 14, 2, 47, 63, 2, 258):
        kn, vn = k[:, pos:pos + n_new], v[:, pos:pos + n_new]
        layer.append(kn, vn, *one, pos, CAPACITY)
        layer.append(kn, vn, *dev, tt.tensor([pos], device="cuda"), CAPACITY, overrun=over)
        for codec, x, buf, kind in ((layer.k_codec, kn, two[0], "k"), (layer.v_codec, vn, two[1], "v")):
            if codec is None:
                tqa.q8_0_append(x, buf, pos, CAPACITY, kind=kind)
            else:
                codec.append(x, buf, pos, CAPACITY, kind=kind)
        pos += n_new
        for a, b, c in zip(one, two, dev):
            assert tt.equal(a, b) and tt.equal(c, b), (pos, n_new)
    assert int(over) == 0
    layer.append(k[:, :9], v[:, :9], *dev, tt.tensor([CAPACITY - 8], device="cuda"), CAPACITY, overrun=over)
    assert int(over) != 0 and all(tt.equal(c, b) for b, c in zip(two, dev))
    with pytest.raises(ValueError):
        layer.append(k[:, :9], v[:, :9], *one, CAPACITY - 8, CAPACITY)
    with pytest.raises(ValueError):
        layer.append(k[:, :1], v[:, :1], one[0], one[1][:-16], 0, CAPACITY)


@pytest.mark.parametrize("fmt", [("q8_0", "turbo3"), ("q8_0", "turbo4"), ("turbo2", "q8_0"), ("turbo4", "q8_0")])
@pytest.mark.parametrize("dtype", ["float16", "float32", "float64"])
@pytest.mark.parametrize("tokens", [1023, 1025, 1152])
def test_prompt_of_a_layer_with_8_bit_rows(fmt, dtype, tokens):
    """64 sequences of 8 and 9 blocks, one launch of the append kernel for K and V: the 8-bit side as
    appended, the turbo side as stored (float16) or appended, sequence by sequence, and nothing past a sequence's last
    block.  (tq_store takes float32 rows as two fp16 terms: no oracle for rows that are computed in 32 bits.)"""
    tt = L.torch()
    n, capacity = 64, 2048
    layer = tqa.LayerKV(tqa.LayerFormat(*fmt))
    gen = tt.Generator("cuda").manual_seed(tokens)
    k, v = (tt.randn((n, tokens, D), generator=gen, device="cuda").to(getattr(tt, dtype)) for _ in range(2))
    caches = [b.fill_(0xA5) for b in layer.new_cache(n, capacity)]
    layer.prefill(k, v, *caches, capacity)
    for codec, x, cache, kind in ((layer.k_codec, k, caches[0], "k"), (layer.v_codec, v, caches[1], "v")):
        blocks = -(-tokens // 128)
        if codec is None:
            want = tqa.q8_0_store(x, kind=kind)[0]
        elif dtype == "float32":
            want = codec.append(x, tt.zeros(n * blocks * O.block_bytes(codec.bits), dtype=tt.uint8, device="cuda"), 0, 128 * blocks, kind=kind)
        else:
            want = codec.store(x, kind=kind)
        got = cache.view(n, capacity // 128, -1)
        assert tt.equal(got[:, :blocks], want.view(n, blocks, -1)), kind
        assert bool((got[:, blocks:] == 0xA5).all()), kind


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("order", ["ascending", "shuffled", "with gaps"])
def test_codes_are_the_number_of_boundaries_below(bits, order):
    """Codebooks in any order, values on, next to and far beyond their boundaries: the code is the count of midpoints of
    neighbouring entries below the value, whatever their order (rows of one non-zero value rotate to +-1/sqrt(128) times it, so
    every rotated value of the row has that size)."""
    rng = np.random.default_rng(bits)
    cent = np.sort(rng.uniform(-0.3, 0.3, 1 << bits))
    if order == "shuffled":
        cent = rng.permutation(cent)
    if order == "with gaps":   # entries of equal value and far outside the rows' range
        cent[: 1 << (bits - 1)] = cent[0] * 100
    codec = tqa.TurboCodec(bits, seed=5, centroids=cent)
    x = rng.standard_normal((1, 384, D))
    x[0, 0], x[0, 1], x[0, 2] = 0, np.eye(D)[7], -3 * np.eye(D)[100]
    cache = L.torch().zeros(tqa.packed_bytes(bits, 1, 384), dtype=L.torch().uint8, device="cuda")
    codec.append(x, cache, 0, 384, kind="k")
    idx = np_(codec.unpack_codes(cache, 1, 384, kind="k")[0])[0].astype(int)
    mid = (cent[1:] + cent[:-1]) / 2
    y = O.rotate_fast(x[0] / np.maximum(np.linalg.norm(x[0], axis=1, keepdims=True), 1e-300), codec.signs1, codec.signs2, D)
    lo, hi = ((mid[None, None] < (y + e)[..., None]).sum(-1) for e in (-2e-6, 2e-6))   # 32-bit rotation of values up to 1
    assert ((idx >= lo) & (idx <= hi)).all()
    assert (lo == hi).mean() > 0.999


@pytest.mark.parametrize("fmt", [("q8_0", "turbo3"), ("turbo4", "q8_0"), ("turbo2", "q8_0")])
@pytest.mark.parametrize("tokens", [128 * 127, 128 * 128])
def test_float32_prompts_keep_their_low_bits(fmt, tokens):
    """Rows of two entries that differ in the last of their 24 bits: half of the rotated values are that difference, on one
    side of the boundary at zero or the other.  Exact in 32-bit sums, whatever the length of the prompt."""
    tt = L.torch()
    layer = tqa.LayerKV(tqa.LayerFormat(*fmt))
    codec, kind = (layer.v_codec, "v") if layer.k_codec is None else (layer.k_codec, "k")
    x = np.zeros((4, tokens, D), np.float32)
    rng = np.random.default_rng(tokens)
    t = np.arange(tokens)
    for s in range(4):
        pair = rng.permuted(np.tile(np.arange(D), (tokens, 1)), axis=1)[:, :2]
        x[s, t, pair[:, 0]], x[s, t, pair[:, 1]] = 1 + 2.0 ** -12 + 2.0 ** -23, 1 + 2.0 ** -12
    xd = tt.from_numpy(x).cuda()
    caches = layer.new_cache(4, tokens)
    layer.prefill(xd, xd, *caches, tokens)
    idx = np_(codec.unpack_codes(caches[kind == "v"], 4, tokens, kind=kind)[0]).astype(int)
    y = O.rotate_fast(x.reshape(-1, D).astype(np.float64), codec.signs1, codec.signs2, D).reshape(x.shape)
    small = np.abs(y) < 1e-6
    assert small.mean() == 0.5 and np.array_equal(idx[small], np.where(y > 0, 1 << (codec.bits - 1), (1 << (codec.bits - 1)) - 1)[small])


@pytest.mark.parametrize("pair", [(2, 2), (3, 3), (4, 4), (4, 2), (4, 3), (3, 2), (2, 4)])
@pytest.mark.parametrize("shape", [(1, 1), (3, 333), (2, 16 * 128), (64, 4 * 128), (64, 4 * 128 + 1)])
@pytest.mark.parametrize("dtype", ["float16", "float32"])
def test_short_prompts_have_the_bytes_of_the_store(pair, shape, dtype):
    """Prompts of up to 256 blocks (and one of 320): K and V in one launch have the bytes of a store per side, into
    buffers of their length and into caches laid out for more tokens."""
    tt = L.torch()
    n, tokens = shape
    kc, vc = (tqa.TurboCodec(b, seed=s) for b, s in zip(pair, (3, 503)))
    k, v = (tt.randn((n, tokens, D), generator=tt.Generator("cuda").manual_seed(s), device="cuda").to(getattr(tt, dtype)) for s in (1, 2))
    k[0, tokens // 2] = 0
    blocks, capacity = -(-tokens // 128), 128 * (-(-tokens // 128) + 3)
    want = kc.store(k, kind="k"), vc.store(v, kind="v")
    assert all(tt.equal(a, b) for a, b in zip(kc.store_kv(vc, k, v), want))
    caches = [tt.full((tqa.packed_bytes(b, n, capacity),), 0xA5, dtype=tt.uint8, device="cuda") for b in pair]
    kc.store_kv(vc, k, v, *caches, capacity=capacity)
    for cache, w in zip(caches, want):
        assert tt.equal(cache.view(n, blocks + 3, -1)[:, :blocks], w.view(n, blocks, -1))
        assert bool((cache.view(n, blocks + 3, -1)[:, blocks:] == 0xA5).all())


@pytest.mark.parametrize("dtype", ["float16", "float32"])
@pytest.mark.parametrize("which", ["k", "v", "both"])
def test_codebooks_that_the_matrix_cores_do_not_take(dtype, which):
    """An asymmetric codebook on one side or both: K and V of a step have the bytes of an append per side, and codes within
    32-bit rounding of the boundaries, with the position on the host and on the device."""
    tt = L.torch()
    cent = np.sort(np.random.default_rng(2).uniform(-0.25, 0.3, 8))
    kc, vc = (tqa.TurboCodec(3, seed=s, centroids=cent if which in (side, "both") else None) for s, side in ((3, "k"), (503, "v")))
    k, v = (tt.randn((N_SEQS, 200, D), generator=tt.Generator("cuda").manual_seed(s), device="cuda").to(getattr(tt, dtype)) for s in (1, 2))
    one, two, dev = ([tt.zeros(tqa.packed_bytes(3, N_SEQS, CAPACITY), dtype=tt.uint8, device="cuda") for _ in range(2)] for _ in range(3))
    pos = 0
    for n_new in (1, 30, 97, 2, 70):
        kn, vn = k[:, pos:pos + n_new], v[:, pos:pos + n_new]
        kc.append_kv(vc, kn, vn, *one, pos, CAPACITY)
        kc.append_kv(vc, kn, vn, *dev, tt.tensor([pos], device="cuda"), CAPACITY)
        kc.append(kn, two[0], pos, CAPACITY, kind="k")
        vc.append(vn, two[1], pos, CAPACITY, kind="v")
        pos += n_new
        for a, b, c in zip(one, two, dev):
            assert tt.equal(a, b) and tt.equal(c, b), (pos, n_new)
    for codec, x, cache, kind in ((kc, k, one[0], "k"), (vc, v, one[1], "v")):
        idx = np_(codec.unpack_codes(cache, N_SEQS, CAPACITY, kind=kind)[0])[:, :200].reshape(-1, D).astype(int)
        xd = np_(x).astype(np.float64).reshape(-1, D)
        y = O.rotate_fast(xd / np.linalg.norm(xd, axis=1, keepdims=True), codec.signs1, codec.signs2, D)
        mid = (codec.centroids[1:] + codec.centroids[:-1]) / 2
        lo, hi = ((mid[None, None] < (y + e)[..., None]).sum(-1) for e in (-1e-6, 1e-6))
        assert ((idx >= lo) & (idx <= hi)).all()


def launches(call):
    """Kernels of a call, as the nodes of its captured graph."""
    tt = L.torch()
    call()
    graph = tt.cuda.CUDAGraph(keep_graph=True)
    with tt.cuda.graph(graph):
        call()
    n = C.c_size_t(0)
    assert L.lib().hipGraphGetNodes(C.c_void_p(graph.raw_cuda_graph()), None, C.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("dtype", ["float16", "float32", "float64"])
@pytest.mark.parametrize("pair", [(2, 2), (3, 3), (4, 4), (4, 2), (4, 3), (3, 2)])
@pytest.mark.parametrize("asymmetric", ["", "k", "v", "kv"])
def test_a_step_is_one_launch(asymmetric, pair, dtype):
    """Whichever codebooks of a layer the matrix cores take: K and V are appended in one launch, with the bytes of an append
    per side."""
    tt = L.torch()
    cent = {b: np.sort(np.random.default_rng(2).uniform(-0.25, 0.3, 1 << b)) for b in pair}
    kc, vc = (tqa.TurboCodec(b, seed=s, centroids=cent[b] if side in asymmetric else None) for b, s, side in zip(pair, (3, 503), "kv"))
    k, v = (tt.randn((N_SEQS, 200, D), generator=tt.Generator("cuda").manual_seed(s), device="cuda").to(getattr(tt, dtype)) for s in (1, 2))
    one, two = ([tt.zeros(tqa.packed_bytes(b, N_SEQS, CAPACITY), dtype=tt.uint8, device="cuda") for b in pair] for _ in range(2))
    for pos, n_new in ((0, 200), (200, 1), (201, 70)):
        kn, vn = k[:, :n_new].contiguous(), v[:, :n_new].contiguous()
        assert launches(lambda: kc.append_kv(vc, kn, vn, *one, pos, CAPACITY)) == 1
        kc.append_kv(vc, kn, vn, *one, pos, CAPACITY)
        kc.append(kn, two[0], pos, CAPACITY, kind="k")
        vc.append(vn, two[1], pos, CAPACITY, kind="v")
        for a, b in zip(one, two):
            assert tt.equal(a, b), (pos, n_new)


@pytest.mark.parametrize("fmt", [("q8_0", "turbo2"), ("q8_0", "turbo3"), ("q8_0", "turbo4"), ("turbo2", "q8_0"), ("turbo3", "q8_0"),
                                 ("turbo4", "q8_0")])
@pytest.mark.parametrize("blocks", [2047, 2048, 3583, 3584])
def test_long_prompt_of_a_layer_with_8_bit_rows(fmt, blocks):
    """The 8-bit side and the turbo side of a long prompt take a launch each from the lengths on where that is the faster, and
    the bytes of a store per side in either way, into caches with room behind them."""
    tt = L.torch()
    layer = tqa.LayerKV(tqa.LayerFormat(*fmt))
    n, per = next((blocks // m, m) for m in (32, 89, 3583) if blocks % m == 0)
    tokens, capacity = 128 * per - 3, 128 * (per + 1)
    gen = tt.Generator("cuda").manual_seed(blocks)
    k, v = (tt.randn((n, tokens, D), generator=gen, device="cuda", dtype=tt.float16) for _ in range(2))
    caches = [b.fill_(0xA5) for b in layer.new_cache(n, capacity)]
    bits = int(max(fmt)[-1])
    assert launches(lambda: layer.prefill(k, v, *caches, capacity)) == (2 if bits == 4 and blocks >= 2048 or bits == 3 and blocks >= 3584 else 1)
    for b in caches:
        b.fill_(0xA5)
    layer.prefill(k, v, *caches, capacity)
    for codec, x, cache, kind in ((layer.k_codec, k, caches[0], "k"), (layer.v_codec, v, caches[1], "v")):
        want = tqa.q8_0_store(x, kind=kind)[0] if codec is None else codec.store(x, kind=kind)
        got = cache.view(n, per + 1, -1)
        assert tt.equal(got[:, :per], want.view(n, per, -1)), kind
        assert bool((got[:, per:] == 0xA5).all()), kind


def near_halves(rng, rows):
    """Rows of four 32-value groups: the literals of test_q8_0_literal_blocks, and per group a scale that is no power of two with
    values on and next to the products that round at a half."""
    x = np.zeros((rows, D), np.float32)
    x[:, :16] = [-127.0, 0.5, -0.5, 1.5, -1.5, 2.5, -2.5, 126.5, -126.5, 0.49999997, -0.49999997, 0.50000006, 3.0, -0.0, 100.25, -100.75]
    for g, amax in enumerate((np.float32(127) * np.float32(1 + 2.0 ** -12), np.float32(100.3), np.float32(0.037)), 1):
        d = amax / np.float32(127)
        half = ((rng.integers(0, 126, (rows, 31)) + 0.5) * float(d)).astype(np.float32)
        half = (half.view(np.int32) + rng.integers(-2, 3, (rows, 31), dtype=np.int32)).view(np.float32)
        x[:, 32 * g:32 * g + 31] = half * rng.choice(np.float32([-1, 1]), (rows, 31))
        x[:, 32 * g + 31] = amax
    return x


@pytest.mark.parametrize("kind", ["k", "v"])
@pytest.mark.parametrize("other", ["q8_0", "turbo3"])
def test_q8_0_rounds_halves_away_from_zero(kind, other):
    """Appends, one side and a layer of any kind, quantise ties and their neighbours as the store and the oracle do."""
    tt = L.torch()
    rows = near_halves(np.random.default_rng(1), 2 * 200).reshape(2, 200, D)
    q, scale = O.q8_0_quantize(rows.reshape(-1, D))
    assert q[0, :16].tolist() == [-127, 1, -1, 2, -2, 3, -3, 127, -127, 0, 0, 1, 3, 0, 100, -101]
    x = tt.from_numpy(rows).cuda()
    layer = tqa.LayerKV(tqa.LayerFormat(*(("q8_0", other) if kind == "k" else (other, "q8_0"))))
    one, (ck, cv) = tt.zeros(2 * 256 * 136, dtype=tt.uint8, device="cuda"), layer.new_cache(2, 256)
    for pos, n_new in ((0, 1), (1, 66), (67, 133)):
        xn = x[:, pos:pos + n_new].contiguous()
        tqa.q8_0_append(xn, one, pos, 256, kind=kind)
        layer.append(xn, xn, ck, cv, pos, 256)
    assert tt.equal(one, ck if kind == "k" else cv)
    assert tt.equal(one, tqa.q8_0_store(x, kind=kind)[0])
    got, s = (np_(a)[:, :200].reshape(400, -1) for a in tqa.q8_0_unpack(one, 2, 256, kind=kind))
    assert np.array_equal(got, q) and np.array_equal(s.astype(np.float16), scale)


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("kind", ["k", "v"])
@pytest.mark.parametrize("dtype", ["float16", "float32"])
def test_infinities_and_nan_stay_in_their_rows(bits, kind, dtype):
    """Rows with an infinity or a NaN have a norm that is not finite; the codes and norms of the tokens that share a word, a
    product or a sum with them are those they have beside ordinary rows, in appends, short prompts and the store."""
    tt = L.torch()
    codec = tqa.TurboCodec(bits, seed=3)
    x = tt.randn((N_SEQS, 400, D), generator=tt.Generator("cuda").manual_seed(bits), device="cuda").to(getattr(tt, dtype))
    bad = x.clone()
    rows = {(0, 0): float("inf"), (0, 7): float("nan"), (0, 130): -float("inf"), (1, 66): float("inf"), (1, 67): float("nan"), (1, 399): -float("inf")}
    for i, ((s, t), value) in enumerate(rows.items()):
        bad[s, t, 37 * i % D] = value
    bad[1, 66, :64], bad[1, 200] = -float("inf"), float("nan")
    whole = np.ones((N_SEQS, 400), bool)
    for s, t in list(rows) + [(1, 200)]:
        whole[s, t] = False

    def appended(r):
        cache = tt.zeros(tqa.packed_bytes(bits, N_SEQS, CAPACITY), dtype=tt.uint8, device="cuda")
        for pos, n_new in ((0, 1), (1, 65), (66, 2), (68, 332)):
            codec.append(r[:, pos:pos + n_new], cache, pos, CAPACITY, kind=kind)
        return codec.unpack_codes(cache, N_SEQS, CAPACITY, kind=kind)

    def prompt(r):
        packed = codec.store_kv(codec, r, r)[kind == "v"]
        return codec.unpack_codes(packed, N_SEQS, 400, kind=kind)

    def stored(r):
        return codec.unpack_codes(codec.store(r, kind=kind), N_SEQS, 400, kind=kind)
    for way in (appended, prompt, stored):
        (codes, norms), (got, g) = ([np_(a)[:, :400] for a in way(r)] for r in (x, bad))
        assert np.array_equal(got[whole], codes[whole]) and np.array_equal(g[whole], norms[whole]), way
        assert not np.isfinite(g[~whole]).any(), way
