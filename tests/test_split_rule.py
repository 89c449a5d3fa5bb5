"""The split count that DecodeAttention takes by itself: the launch plan it estimates with is the library's, and the count
stays where the estimate does not clearly favour another."""
import ctypes as C
import itertools

import pytest

from turboquant_plus_amd import _lib as L
from turboquant_plus_amd import turbo as T


def align(n):
    return (n + 255) // 256 * 256


@pytest.mark.parametrize("k8,v8", itertools.product((False, True), repeat=2))
@pytest.mark.parametrize("per_kv", [1, 4, 8])
def test_plan_is_the_library_s(k8, v8, per_kv):
    """tq_attn_workspace_bytes makes room for the partials of a call with and without a bias list, whichever are more:
    the number of partials per group (a bias list runs the eight-head variant without its workgroups of twelve)."""
    eight, rest = per_kv > 4, set()
    for kv_heads, batch, n in itertools.product((1, 3, 8), (1, 2, 6, 20), (1, 2, 4) + T._SPLIT_COUNTS + (60, 144, 464)):
        groups = kv_heads * batch
        p = L.TQAttnParams(batch=batch, n_q_heads=per_kv * kv_heads, n_kv_heads=kv_heads, tokens=70000, n_splits=n,
                           k_format=L.KFMT_Q8_0 if k8 else L.KFMT_TURBO, v_format=L.KFMT_Q8_0 if v8 else L.KFMT_TURBO, scale=1.0, head_dim=128)
        parts = groups * max(T._workgroups(n, groups, eight, tk, not v8)[1] for tk in {not k8, False})
        rows = 8 if eight else 4
        room = align(parts * rows * 512) + align(parts * rows * 8) + 2 * align(parts * 8)
        rest.add(L.lib().tq_attn_workspace_bytes(C.byref(p)) - room)
    assert len(rest) == 1 and rest.pop() >= 0   # what does not depend on the shape


def test_rule():
    four, eight = dict(eight_heads=False, turbo_k=True, turbo_v=True), dict(eight_heads=True, turbo_k=True, turbo_v=True)
    for groups, tokens in ((128, 32768), (32, 32768), (8, 32768), (8, 131072), (64, 8192), (512, 2048)):
        d = T.default_splits(groups, tokens)
        assert T.balanced_splits(groups, tokens, d, **four) == d           # the shapes the default was swept at
    assert T.balanced_splits(8, 4000, 16, **four) == 32
    assert T.balanced_splits(40, 25000, 48, **eight) < 48
    for groups, tokens, kw in itertools.product((1, 2, 7, 40, 300, 5000), (1, 63, 64, 700, 5000, 90000, 3_000_000), (four, eight)):
        d = T.default_splits(groups, tokens, eight_heads=kw["eight_heads"])
        n = T.balanced_splits(groups, tokens, d, **kw)
        assert n == d or (n in T._SPLIT_COUNTS and 2 * n <= (tokens + 63) // 64 + 2)


def test_room_for_the_table_and_plan_of_a_bias_list():
    four, eight = dict(eight_heads=False, turbo_k=True, turbo_v=True), dict(eight_heads=True, turbo_k=True, turbo_v=True)
    # 1000 workgroups of four: four fit a CU, three beside a 32 KB table (8 splits: 25.7 us, 20: 31.3)
    assert T.balanced_splits(200, 3175, 8, **four) == 20
    assert T.balanced_splits(200, 3175, 8, three_bit=True, **four) == 8
    # without workgroups of twelve 36 splits are 360 workgroups of four (48: 49.8 us, 36: 58.0)
    assert T.balanced_splits(40, 27579, 48, **eight) == 36
    assert T.balanced_splits(40, 27579, 48, bias_list=True, **eight) == 48
    # a workgroup of four per CU with Sparse V (32: 38.8 us, 20: 44.7) or a list; without, at 29 700 tokens, 55.3 and 48.0
    q8v = dict(eight_heads=False, turbo_k=True, turbo_v=False, three_bit=True)
    assert T.balanced_splits(48, 18060, 32, **q8v) == 20
    assert T.balanced_splits(48, 18060, 32, sparse_v=True, **q8v) == T.balanced_splits(48, 18060, 32, bias_list=True, **q8v) == 32
