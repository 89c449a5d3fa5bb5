"""Which kernel the decode attention's launcher takes, on both sides of every edge of its rule (tq_decode_attention_plan, host
only), and that the shapes of the GPU tests lie on the sides that they are there for."""
import ctypes as C

import pytest

from turboquant_plus_amd import _lib as L


def plan(k, v, batch, heads, kv_heads, tokens, n_splits, *, one_table=None, dense=False, entries=0, tau=0.0, head_dim=128, workspace=None):
    p = L.TQAttnParams(batch=batch, n_q_heads=heads, n_kv_heads=kv_heads, tokens=tokens, n_splits=n_splits, scale=1.0, sparse_v_tau=tau,
                       k_format=L.KFMT_Q8_0 if k == 8 else L.KFMT_TURBO, v_format=L.KFMT_Q8_0 if v == 8 else L.KFMT_TURBO,
                       bias_entries=entries, head_dim=head_dim)
    out = L.TQAttnPlan()
    if workspace is None:
        workspace = L.lib().tq_attn_workspace_bytes(C.byref(p))
    L.check(L.lib().tq_decode_attention_plan(C.byref(p), k, v, k == v if one_table is None else one_table, dense, workspace, C.byref(out)))
    return out


def lanes(*args, **kw):
    return bool(plan(*args, **kw).lane_tables)


def test_a_side_of_4_bit_codes_with_128_dims():
    shape = (2, 8, 2, 4096, 8)
    assert all(lanes(k, v, *shape) for k, v in ((4, 4), (4, 2), (4, 3), (3, 4), (2, 4)))
    assert not any(lanes(k, v, *shape) for k, v in ((2, 2), (3, 3), (2, 3), (3, 2), (8, 4), (4, 8), (8, 8)))
    assert not lanes(4, 4, *shape, head_dim=256)


@pytest.mark.parametrize("G", [4, 8])
def test_three_tiles_per_wavefront(G):
    at = lambda tokens, splits: lanes(4, 4, 2, 2 * G, 2, tokens, splits)
    assert at(8 * 64 + 1, 4) and not at(8 * 64, 4)
    assert at(12 * 64 - 27, 4) and at(16 * 64 + 1, 8) and not at(16 * 64, 8)


@pytest.mark.parametrize("G", [4, 8])
def test_four_wavefronts_per_workgroup(G):
    for n, want in ((4, 4), (2, 2), (6, 2), (1, 1)):
        p = plan(4, 4, 2, 2 * G, 2, 64 * 64, n)
        assert p.wavefronts == want and bool(p.lane_tables) == (want >= 4)


def test_room_for_the_tables_beside_each_other():
    """67 KB for a workgroup of four wavefronts with one table: two to a CU."""
    for groups, n, workgroups, want in ((100, 20, 500, True), (103, 20, 515, False), (200, 8, 400, True), (200, 20, 1000, False)):
        p = plan(4, 4, groups, 4, 1, 3175, n)
        assert (p.wavefronts, p.workgroups) == (n * groups // workgroups, workgroups) and bool(p.lane_tables) == want, (groups, n)
    # 128 KB for two tables: a workgroup per CU
    assert lanes(4, 4, 64, 4, 1, 32768, 32, one_table=False) and not lanes(4, 4, 128, 4, 1, 32768, 24, one_table=False)
    # 96 KB: 320 workgroups of eight heads have no room
    assert not lanes(4, 3, 20, 64, 8, 2500, 8) and lanes(4, 3, 16, 64, 8, 2500, 8)


def test_bias():
    four, eight = (2, 8, 2, 4096, 8), (2, 16, 2, 4096, 8)
    for tau in (0.0, 1e-3):
        assert lanes(4, 4, *eight, entries=16, tau=tau) and not lanes(4, 4, *four, entries=16, tau=tau)
        assert not lanes(4, 4, *eight, dense=True, tau=tau) and not lanes(4, 4, *four, dense=True, tau=tau)
        assert lanes(4, 4, *eight, tau=tau) and lanes(4, 4, *four, tau=tau)


def test_passes_share_a_launch_and_the_room():
    one, two = plan(4, 4, 20, 8, 1, 32768, 64), plan(4, 4, 20, 16, 1, 32768, 64)
    assert (one.passes, two.passes) == (1, 2) and two.workgroups == 2 * one.workgroups
    assert plan(4, 4, 20, 16, 1, 32768, 64, tau=1e-3).passes == 1
    assert plan(4, 4, 20, 16, 1, 32768, 64, workspace=L.lib().tq_attn_workspace_bytes(
        C.byref(L.TQAttnParams(batch=20, n_q_heads=8, n_kv_heads=1, tokens=32768, n_splits=64, scale=1.0, head_dim=128)))).passes == 1
    # 80 splits of 20 groups: 400 workgroups of four in a pass, two to a CU; both passes are 800
    assert lanes(4, 4, 20, 8, 1, 32768, 80) and not lanes(4, 4, 20, 16, 1, 32768, 80)


@pytest.mark.parametrize("k,v", [(4, 4), (4, 2), (4, 3), (3, 4), (2, 4)])
def test_shapes_of_the_gpu_tests(k, v):
    """tests/test_gpu_attention_turbo4.py: which of its steps run the kernel that it is about."""
    for G in (1, 4, 5, 8, 12):
        assert [lanes(k, v, 2, 2 * G, 2, N, n) for N, n in ((12 * 64 - 27, 4), (8 * 64, 4), (17 * 64 + 1, 8))] == [True, False, True]
    for G, entries, tau in ((8, 21, 0.0), (8, 0, 1e-3), (7, 21, 1e-3), (4, 0, 1e-3)):
        assert lanes(k, v, 2, 2 * G, 2, 14 * 64 + 3, 4, entries=entries, tau=tau)
    assert not lanes(k, v, 2, 8, 2, 14 * 64 + 3, 4, entries=21, tau=1e-3)
    if k == v:
        assert lanes(4, 4, 3, 4, 1, 16 * 64 - 5, 4, one_table=False) and lanes(4, 4, 3, 8, 1, 16 * 64 - 5, 4, one_table=False)
    assert lanes(4, 4, 1, 16, 2, 40 * 64, 8)


def test_bad_arguments():
    with pytest.raises(ValueError):
        plan(5, 4, 1, 4, 1, 128, 1)
    with pytest.raises(ValueError):
        plan(4, 4, 1, 4, 1, 128, 1, entries=-1)
    p = L.TQAttnParams(batch=1, n_q_heads=4, n_kv_heads=1, tokens=128, n_splits=1, scale=1.0, head_dim=128)
    assert L.lib().tq_decode_attention_plan(C.byref(p), 4, 4, 1, 0, 0, None) == L.ERR_ARG
    assert L.lib().tq_decode_attention_plan(None, 4, 4, 1, 0, 0, C.byref(L.TQAttnPlan())) == L.ERR_ARG
