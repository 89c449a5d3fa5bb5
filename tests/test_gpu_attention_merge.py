"""The end of a decode step: the wavefronts' results of a workgroup, the workgroups' partials of a group, and the counter that
picks the workgroup which merges them, at every number of wavefronts per workgroup that the launch plan makes."""
import numpy as np
import pytest

import turboquant_plus_amd as tqa
from turboquant_plus_amd import _lib as L
from test_gpu_attention import D, assert_close, make_kv, np_, reference_attention

pytestmark = pytest.mark.gpu


# (query heads per KV head, groups, splits) -> wavefronts per workgroup, partials per group:
# four heads 1 x 3, 2 x 3, 4 x 3, 8 x 3 (and x 1), 16 x 2, 16 x 17; one partial: one group and four groups to a workgroup
# eight heads 1 x 5, 2 x 1, 3 x 4, 4 x 8, 4 x 11, 6 x 2, 8 x 1, 12 x 1; two groups of four wavefronts to a workgroup
@pytest.mark.parametrize("G,groups,n_splits", [(4, 6, 3), (4, 6, 6), (4, 6, 12), (4, 90, 24), (4, 256, 8), (4, 128, 32), (4, 20, 272), (4, 300, 1),
                                               (3, 1024, 4), (8, 6, 5), (7, 300, 2), (8, 6, 12), (8, 6, 32), (5, 6, 44), (8, 150, 12), (8, 256, 8),
                                               (8, 256, 12), (6, 512, 4)])
def test_every_shape_of_the_merge(G, groups, n_splits):
    N = 64 * min(n_splits, 24) - 27
    k, v, kc, vc, kp, vp = make_kv(1, groups, N, seed=groups + n_splits)
    q = np.random.default_rng(n_splits).standard_normal((1, G * groups, D)).astype(np.float16)
    attn = tqa.DecodeAttention(kc, vc, 1, G * groups, groups, N, n_splits=n_splits, poison_output=True)
    # whatever a fresh workspace holds is neither a count nor a partial
    attn.workspace.random_(0, 256)
    first = attn(q, kp, vp).clone()
    for _ in range(3):
        again = attn(q, kp, vp)
        assert bool((again == first).all())
    sel = slice(0, groups) if groups <= 20 else slice(groups - 12, groups)    # the last groups: past the first round of workgroups
    n_sel = sel.stop - sel.start
    per_k, per_v = kp.numel() // groups, vp.numel() // groups
    ref, _, _ = reference_attention(q[:, G * sel.start:], kc, vc, kp[per_k * sel.start:], vp[per_v * sel.start:], 1, G * n_sel, n_sel, N,
                                    1 / np.sqrt(D))
    assert_close(np_(first)[:, G * sel.start:], ref)


def test_steps_captured_in_a_graph_find_their_counters():
    """The tag of a captured launch is the same at every replay, and eager calls on the same workspace come in between."""
    tt = L.torch()
    N, groups = 1500, 5
    k, v, kc, vc, kp, vp = make_kv(1, groups, N, seed=5)
    q = tt.from_numpy(np.random.default_rng(3).standard_normal((1, 8 * groups, D)).astype(np.float16)).cuda()
    attn = tqa.DecodeAttention(kc, vc, 1, 8 * groups, groups, N, n_splits=16)
    want = attn(q, kp, vp).clone()
    tt.cuda.synchronize()
    graph = tt.cuda.CUDAGraph()
    with tt.cuda.graph(graph):
        attn(q, kp, vp)
    for step in range(6):
        attn.out.fill_(float("nan"))
        graph.replay()
        assert bool((attn.out == want).all()), step
        if step % 2:
            attn.out.fill_(float("nan"))
            assert bool((attn(q, kp, vp) == want).all()), step


@pytest.mark.parametrize("G,n_splits,bits", [(4, 4, 3), (4, 32, 3), (8, 4, 4), (8, 12, 3), (8, 32, 4)])
def test_a_split_whose_sum_is_not_a_number(G, n_splits, bits):
    """A logit of +inf (a K row whose norm is beyond fp16) makes the sum of its wavefront's weights NaN.  With Sparse V, which skips
    weights that are not above the threshold, that wavefront has nothing to add, and its workgroup's others count as they do without it."""
    tt = L.torch()
    tiles, groups = 4 * n_splits, 3
    N = 64 * tiles
    k, v, kc, vc, kp, vp = make_kv(1, groups, N, seed=bits, kbits=bits, vbits=bits)
    q = np.random.default_rng(7).standard_normal((1, G * groups, D)).astype(np.float16)
    q[:] = q[:, :1]                                     # one query for all heads: the logit's sign is the same for each
    big = k.astype(np.float32)
    big[1, 0] = 1e6 * q[0, 0].astype(np.float32) / np.linalg.norm(q[0, 0].astype(np.float32))
    assert np.linalg.norm(big[1, 0]) > np.finfo(np.float16).max
    kp2 = kc.store(big, kind="k")
    attn = tqa.DecodeAttention(kc, vc, 1, G * groups, groups, N, n_splits=n_splits, sparse_v_tau=1e-6, poison_output=True)
    got = np_(attn(q, kp2, vp)).copy()
    per_k, per_v = kp.numel() // groups, vp.numel() // groups
    # the group without its first split: what the other wavefronts have
    cut = 64 * 4
    rest_k, rest_v = kc.store(k[1:2, cut:], kind="k"), vc.store(v[1:2, cut:], kind="v")
    ref, _, _ = reference_attention(q[:, G:2 * G], kc, vc, rest_k, rest_v, 1, G, 1, N - cut, 1 / np.sqrt(D))
    assert np.isfinite(got).all()
    assert_close(got[:, G:2 * G], ref)
    others = np_(attn(q, kc.store(k.astype(np.float32), kind="k"), vp))     # fp32 rows, as above
    assert np.array_equal(got[:, :G], others[:, :G]) and np.array_equal(got[:, 2 * G:], others[:, 2 * G:])
