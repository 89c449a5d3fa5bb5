"""Host-array handling of the NumPy classes that needs no GPU."""
import numpy as np
import pytest

from turboquant_plus_amd.kv_cache import _joined


@pytest.mark.parametrize("t", [0, 1, 4])
def test_one_token_pieces_of_a_token_major_container(t):
    """A piece of one token is contiguous whatever the stride of its token axis: heads of one token in containers
    [tokens, heads, d] and [tokens, heads] are neighbours in memory whose stride along tokens is not theirs to use."""
    x = np.arange(60).reshape(5, 3, 4)
    joined = _joined([x[t:t + 1, h] for h in range(3)])
    assert joined.flags.c_contiguous and np.array_equal(joined, x[t])
    norms = np.arange(15.0).reshape(5, 3)
    assert np.array_equal(_joined([norms[t:t + 1, h] for h in range(3)]), norms[t])
    one = np.arange(4.0).reshape(1, 4)
    assert np.array_equal(_joined([one[:, h] for h in range(4)]), one[0])


def test_joined_equals_concatenate():
    """Pieces of one array, neighbours or not, in any order and of any axis order."""
    x = np.random.default_rng(0).standard_normal((2, 3, 5, 4))
    for a in (x, x.transpose(1, 0, 2, 3), x.transpose(2, 1, 0, 3), x[::-1], x[:, :, ::2], x[..., ::-1], x[:, :, :1], np.asfortranarray(x)):
        for pieces in ([a[i, j] for i in range(a.shape[0]) for j in range(a.shape[1])], [a[i, 0] for i in range(a.shape[0])],
                       [a[0, 0], a[0, 0]], [a[0, 0]], [a[0, 0], a[0, 1].astype(np.float32)]):
            assert np.array_equal(_joined(pieces), np.concatenate(pieces, axis=0))


def test_scalar_norms_join():
    """Containers of one token may hold a plain number per (layer, head)."""
    for scalars in ([np.float64(2.5), 3, np.array(4.0)], list(np.arange(3.0)[:, None].T.reshape(3))):
        assert np.array_equal(_joined(scalars), np.asarray(scalars, dtype=np.float64))
    z = np.arange(3.0)
    assert np.array_equal(_joined([z[i:i + 1].reshape(()) for i in range(3)]), z)
