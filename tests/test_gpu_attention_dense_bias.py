"""Dense bias rows where their variants are short of registers (eight heads in workgroups of twelve wavefronts), with
a list beside them, and with the split counts that an object takes by itself."""
import numpy as np
import pytest

import turboquant_plus_amd as tqa
from turboquant_plus_amd import _lib as L
from test_gpu_attention import D, assert_close, make_kv, np_, reference_attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("kbits,vbits", [(2, 2), (3, 3), (4, 4), (4, 2), (3, 4), (2, 3)])
def test_eight_heads_in_workgroups_of_twelve(kbits, vbits, sparse):
    """24 splits of 140 groups: twelve wavefronts per workgroup, two partials per group; rows that allow 16-byte loads and others."""
    tt = L.torch()
    groups, G = 140, 8
    for N in (24 * 64, 24 * 64 - 29):
        k, v, kc, vc, kp, vp = make_kv(1, groups, N, seed=N + kbits, kbits=kbits, vbits=vbits)
        rng = np.random.default_rng(vbits)
        q = rng.standard_normal((1, G * groups, D)).astype(np.float16)
        bias = rng.uniform(-2.0, 2.0, (1, G * groups, N)).astype(np.float32)
        bias[:, ::3, N - 1] = 6.0
        bias[:, 1::3, 0] = -np.inf
        bd = tt.from_numpy(bias).cuda()
        tau = 1e-3 if sparse else 0.0
        attn = tqa.DecodeAttention(kc, vc, 1, G * groups, groups, N, n_splits=24, sparse_v_tau=tau, poison_output=True)
        out = np_(attn(q, kp, vp, bias=bd)).copy()
        part = bias * (rng.random(bias.shape) < 0.999)
        part[bias == -np.inf] = -np.inf
        lists = tqa.sparse_bias_from_dense(np.where(part == bias, np.float32(0), bias))
        both = np_(attn(q, kp, vp, bias=tt.from_numpy(part).cuda(), sparse_bias=lists))
        at = slice(groups - 6, groups)
        per_k, per_v = kp.numel() // groups, vp.numel() // groups
        ref, _, _ = reference_attention(q[:, G * at.start:], kc, vc, kp[per_k * at.start:], vp[per_v * at.start:], 1, 6 * G, 6, N, 1 / np.sqrt(D),
                                        n_splits=24, tau=tau, bias=bias[:, G * at.start:])
        assert_close(out[:, G * at.start:], ref)
        assert_close(both[:, G * at.start:], ref)


def test_each_call_takes_its_own_split_count():
    """One object, calls without a bias, with dense rows, with a list and with both, in turn: counts differ, the workspace has
    room for each, results hold."""
    tt = L.torch()
    groups, G, N = 36, 4, 1731
    k, v, kc, vc, kp, vp = make_kv(1, groups, N, seed=9, kbits=4, vbits=4)
    rng = np.random.default_rng(1)
    q = rng.standard_normal((1, G * groups, D)).astype(np.float16)
    bias = np.where(rng.random((1, G * groups, N)) < 0.01, np.float32(3), np.float32(0))
    bd, lists = tt.from_numpy(bias).cuda(), tqa.sparse_bias_from_dense(bias)
    attn = tqa.DecodeAttention(kc, vc, 1, G * groups, groups, N, poison_output=True)
    ref = [reference_attention(q, kc, vc, kp, vp, 1, G * groups, groups, N, 1 / np.sqrt(D), bias=b)[0] for b in (None, bias, 2 * bias)]
    seen = []
    for _ in range(2):
        for kw, want in (({}, ref[0]), (dict(bias=bd), ref[1]), (dict(sparse_bias=lists), ref[1]), (dict(bias=bd, sparse_bias=lists), ref[2])):
            assert_close(np_(attn(q, kp, vp, **kw)), want)
            seen.append(attn.params.n_splits)
    assert seen[:4] == seen[4:] == [*(attn._own_splits[i] for i in (0, 2, 1, 1))] and seen[0] != seen[1]
