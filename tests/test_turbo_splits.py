"""The split count of steps on turbo rows: the launch plan's counts, taken where they are clearly ahead."""
import itertools

import pytest

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
