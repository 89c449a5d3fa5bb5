"""The split count of steps on turbo rows: the launch plan's counts, taken where they are clearly ahead."""
import itertools
import math
import random
from types import SimpleNamespace

import numpy as np
import pytest

from test_attention_plan import plan
from turboquant_plus_amd import turbo as T


@pytest.mark.parametrize("eight", [False, True])
@pytest.mark.parametrize("k,v", [(2, 2), (3, 3), (3, 2), (4, 4), (4, 2), (3, 4)])
def test_counts(k, v, eight):
    for groups, tokens, one in itertools.product((1, 2, 7, 40, 300, 5000), (1, 63, 64, 700, 5000, 90000, 3_000_000), {k == v, False}):
        now = T.balanced_splits(groups, tokens, T.default_splits(groups, tokens, eight_heads=eight), eight_heads=eight, turbo_k=True, turbo_v=True)
        n = T.turbo_splits(groups, tokens, now, k_bits=k, v_bits=v, one_table=one, eight_heads=eight)
        assert n == now or (n in T._SPLIT_COUNTS and n <= (tokens + 63) // 64 and (not eight or groups <= 256))


def test_shapes_that_were_timed():
    four, eight = dict(eight_heads=False), dict(eight_heads=True)
    assert T.turbo_splits(36, 1731, 8, k_bits=3, v_bits=4, one_table=False, **four) == 28     # 15.0 us with 8, 9.4 with 28
    assert T.turbo_splits(32, 1747, 8, k_bits=3, v_bits=3, one_table=True, **four) == 28      # 12.0 and 8.8
    assert T.turbo_splits(16, 1781, 8, k_bits=4, v_bits=4, one_table=True, **eight) == 28     # 14.9 and 9.7
    assert T.turbo_splits(16, 1740, 8, k_bits=3, v_bits=3, one_table=True, **eight) == 28     # 14.4 and 9.9
    # workgroups of four, five to a CU: 15 % slower than the estimate has them
    assert T.turbo_splits(288, 3676, 8, k_bits=4, v_bits=4, one_table=True, **eight) == 8
    for bits in (2, 3, 4):
        assert T.turbo_splits(128, 32768, 32, k_bits=bits, v_bits=bits, one_table=True, **four) == 32
    assert T.turbo_splits(8, 32768, 256, k_bits=3, v_bits=3, one_table=True, **four) == 256


def _shapes(eight):
    rng = random.Random(11 + eight)
    for _ in range(1500):
        k, v = rng.choice([(2, 2), (3, 3), (4, 4), (4, 2), (3, 4), (4, 3), (2, 4)])
        per_kv = rng.choice((5, 8, 12, 16, 24)) if eight else rng.choice((1, 3, 4))
        yield (rng.choice((1, 2, 8)), int(math.exp(rng.uniform(0, math.log(300)))), per_kv, int(math.exp(rng.uniform(math.log(200), math.log(131072)))),
               k, v, k == v and rng.random() < 0.7, rng.choice(T._SPLIT_COUNTS))


@pytest.mark.parametrize("eight", [False, True])
def test_estimates_are_made_for_the_kernel_that_is_launched(eight):
    """The estimate's workgroups and its choice of a kernel are the launcher's, also where several passes share a launch."""
    taken = 0
    for kv_heads, batch, per_kv, tokens, k, v, one, n in _shapes(eight):
        p = plan(k, v, batch, per_kv * kv_heads, kv_heads, tokens, n, one_table=one)
        waves, parts, wgs = T._workgroups(n, batch * kv_heads, eight, True, True)
        passes = -(-per_kv // 8) if eight else 1
        assert (p.wavefronts, p.partials, p.workgroups, p.passes) == (waves, parts, wgs * passes, passes)
        lds = T._lane_tables(k, v, one, eight, n, waves, wgs * passes, (tokens + 63) // 64)
        assert bool(p.lane_tables) == bool(lds)
        taken += bool(lds)
    assert taken > 100


def test_steps_of_several_passes():
    """us with both counts, measured."""
    turbo3 = dict(k_bits=3, v_bits=3, one_table=True, eight_heads=True)
    assert T.turbo_splits(104, 1750, 8, passes=3, **turbo3) == 8      # 25.2; 28 splits 41.1
    assert T.turbo_splits(96, 1769, 8, passes=2, **turbo3) < 28       # 8: 19.0; 28: 27.9
    turbo4 = dict(k_bits=4, v_bits=4, one_table=True, eight_heads=True)
    assert T.turbo_splits(20, 32768, 72, passes=2, **turbo4) != 80    # no room for the tables of both passes' workgroups


def test_every_kind_of_call_has_its_own_count():
    """Dense bias rows run in the general kernel; us with the counts, measured."""
    codec = lambda bits, scale=1.0: SimpleNamespace(bits=bits, centroids=scale * np.arange(1 << bits))
    four, three = codec(4), codec(3)
    none, listed, dense = T.call_splits(four, three, 288, 4, 1246)
    assert (none, listed, dense) == (20, 8, 8)                          # dense: 8 20.6, 20 26.0
    assert T.call_splits(four, three, 40, 8, 41753)[2] == 36            # 36 71.7, 20 89.9
    assert T.call_splits(codec(2), codec(2), 192, 8, 4081)[2] < 32      # 8 32.1, 32 39.5
    assert T.call_splits(four, codec(2), 128, 4, 38329)[2] == 32        # 32 98, 8 159
    for k, v, per_kv, dim in itertools.product((None, three, four), (None, three, four), (1, 4, 8, 16), (128, 256)):
        for groups, tokens in ((3, 900), (16, 1781), (40, 27600)):
            for sparse in (False, True):
                none, listed, dense = T.call_splits(k, v, groups, per_kv, tokens, head_dim=dim, sparse_v=sparse)
                if sparse or dim == 256 or k is None or v is None:
                    assert none == dense
                elif k is v is four and per_kv <= 4:
                    assert dense == listed


def test_outside_of_what_was_fitted():
    """us with both counts, measured."""
    four = dict(eight_heads=False)
    assert T.turbo_splits(831, 795, 2, k_bits=4, v_bits=2, one_table=False, **four) == 2        # 21.9; 8 splits 27.2
    assert T.turbo_splits(853, 682, 2, k_bits=4, v_bits=4, one_table=True, **four) == 2         # 24.1; 8: 29.8
    for tokens in (318860, 325710):
        assert T.turbo_splits(1, tokens, 2048, k_bits=4, v_bits=4, one_table=True, eight_heads=True) == 2048    # 40; 256: 48
    rng = random.Random(3)
    for _ in range(2000):
        groups, tokens = rng.randint(301, 1100), int(math.exp(rng.uniform(math.log(400), math.log(131072))))
        k, v = rng.choice([(2, 2), (3, 3), (3, 2), (4, 4), (4, 2), (4, 3), (3, 4)])
        now = T.balanced_splits(groups, tokens, T.default_splits(groups, tokens), turbo_k=True, turbo_v=True, three_bit=3 in (k, v), **four)
        n = T.turbo_splits(groups, tokens, now, k_bits=k, v_bits=v, one_table=k == v, **four)
        if n != now:    # few shapes of the others gained
            p = plan(k, v, groups, 4, 1, tokens, n)
            assert p.lane_tables and -(-tokens // 64) >= 5 * n + 1
