"""Decode steps with 4-bit rows on a side, where the look-up tables have a copy per lane: every pair of widths, four and eight
heads per pass, Sparse V and bias lists, at the edges of the rule that takes them (three tiles per wavefront, four wavefronts
per workgroup, room for the tables) against the oracle on the stored codes.  Which of them run that kernel is checked in
test_attention_plan.py."""
import numpy as np
import pytest

import tq_oracle as O
import turboquant_plus_amd as tqa
from turboquant_plus_amd import _lib as L
from test_gpu_attention import D, assert_close, make_kv, np_, reference_attention

pytestmark = pytest.mark.gpu
PAIRS = [(4, 4), (4, 2), (4, 3), (3, 4), (2, 4)]


@pytest.mark.parametrize("G", [1, 4, 5, 8, 12])
@pytest.mark.parametrize("kbits,vbits", PAIRS)
def test_every_pair_of_widths(kbits, vbits, G):
    # tiles per wavefront: 3 with a ragged last tile, 2 (the general variant), 3 with splits that have no tile at all
    for seed, (N, n_splits) in enumerate([(12 * 64 - 27, 4), (8 * 64, 4), (17 * 64 + 1, 8)]):
        k, v, kc, vc, kp, vp = make_kv(2, 2, N, seed=10 * kbits + seed, kbits=kbits, vbits=vbits)
        q = np.random.default_rng(seed).standard_normal((2, 2 * G, D)).astype(np.float16)
        attn = tqa.DecodeAttention(kc, vc, 2, 2 * G, 2, N, n_splits=n_splits, poison_output=True)
        ref, _, _ = reference_attention(q, kc, vc, kp, vp, 2, 2 * G, 2, N, 1 / np.sqrt(D))
        assert_close(np_(attn(q, kp, vp)), ref)


@pytest.mark.parametrize("G", [4, 8])
def test_two_tables_of_64_kb(G):
    """4-bit codebooks that differ between K and V: 128 KB of tables, a workgroup per CU."""
    N = 16 * 64 - 5
    rng = np.random.default_rng(G)
    k, v = (rng.standard_normal((3, N, D)).astype(np.float16) for _ in range(2))
    kc = tqa.TurboCodec(4, seed=42)
    vc = tqa.TurboCodec(4, seed=542, centroids=1.07 * np.asarray(kc.centroids))
    kp, vp = kc.store(k, kind="k"), vc.store(v, kind="v")
    q = rng.standard_normal((3, G, D)).astype(np.float16)
    ref, _, _ = reference_attention(q, kc, vc, kp, vp, 3, G, 1, N, 1 / np.sqrt(D))
    assert_close(np_(tqa.DecodeAttention(kc, vc, 3, G, 1, N, n_splits=4, poison_output=True)(q, kp, vp)), ref)


@pytest.mark.parametrize("kbits,vbits", PAIRS)
@pytest.mark.parametrize("G,listed,sparse", [(8, True, False), (8, False, True), (7, True, True), (4, False, True), (4, True, True)])
def test_sparse_v_and_bias_lists(kbits, vbits, G, listed, sparse):
    B, Hkv, N, n_splits, E = 2, 2, 14 * 64 + 3, 4, 21
    tt = L.torch()
    k, v, kc, vc, kp, vp = make_kv(B, Hkv, N, seed=vbits, kbits=kbits, vbits=vbits)
    rng = np.random.default_rng(G)
    q = rng.standard_normal((B, G * Hkv, D)).astype(np.float16)
    bias = np.zeros((B, G * Hkv, N), np.float32)
    for b in range(B):
        for h in range(G * Hkv):
            # a head without entries, one with a run of them, the others spread, the last token among them
            at = [] if h == 1 else range(70, 70 + E) if h == 2 else np.r_[rng.choice(N - 1, E - 1, replace=False), N - 1]
            bias[b, h, list(at)] = 4.0
    lists = tqa.sparse_bias_from_dense(tt.from_numpy(bias).cuda()) if listed else None
    tau = 1e-3 if sparse else 0.0
    attn = tqa.DecodeAttention(kc, vc, B, G * Hkv, Hkv, N, n_splits=n_splits, sparse_v_tau=tau, poison_output=True)
    out = np_(attn(q, kp, vp, sparse_bias=lists))
    ref, skip, _ = reference_attention(q, kc, vc, kp, vp, B, G * Hkv, Hkv, N, 1 / np.sqrt(D), n_splits=n_splits, tau=tau,
                                       bias=bias if listed else None)
    assert_close(out, ref)
    if sparse:
        assert abs(attn.skip_rate() - skip) < 1e-3


def test_context_length_read_from_memory():
    """One captured length for a growing cache: splits without tiles, a ragged tile, a length of zero tiles for most wavefronts."""
    tt = L.torch()
    N, G = 40 * 64, 8
    k, v, kc, vc, kp, vp = make_kv(1, 2, N, seed=3, kbits=4, vbits=4)
    q = np.random.default_rng(5).standard_normal((1, 2 * G, D)).astype(np.float16)
    now = tt.zeros(1, dtype=tt.int64, device="cuda")
    attn = tqa.DecodeAttention(kc, vc, 1, 2 * G, 2, N, n_splits=8, tokens_on_device=now, poison_output=True)
    for t in (N, N - 1, 700, 65, 1):
        now.fill_(t)
        ref, _, _ = reference_attention(q, kc, vc, kp, vp, 1, 2 * G, 2, t, 1 / np.sqrt(D), capacity=N)
        assert_close(np_(attn(q, kp, vp)), ref)
