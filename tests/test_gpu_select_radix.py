"""The selection's radix passes, which take the calls whose bracket misses the
rank: the smallest values lie exactly where the first sample is taken, so the
bracket of any larger rank is far below it.  (Ties alone do not send a call
there: the bracket orders by value and index.)  With distinct values the passes
go over the keys, with ties over the indices too; the workspace then holds what
the narrowing left."""
import numpy as np
import pytest

from multilanguagekdtree_amd import _lib
from multilanguagekdtree_amd import kdtree as K

SAMPLE = 8192


def sampled(n):
    """The positions of the first sample (sample_at in kd_select.hip)."""
    i = np.arange(SAMPLE, dtype=np.uint64)
    m, c = np.uint64(0xFFFFFFFF), np.uint64(0x9E3779B1)
    x = (i + np.uint64(1)) * c & m
    x = (x ^ x >> np.uint64(15)) * c & m
    x = (x ^ x >> np.uint64(13)) * c & m
    x ^= x >> np.uint64(16)
    n = np.uint64(n)
    first = i * n // np.uint64(SAMPLE)
    size = (i + np.uint64(1)) * n // np.uint64(SAMPLE) - first
    return (first + (x * size >> np.uint64(32))).astype(np.int64)


def inputs(n, kind, seed):
    """Indices in random order and values such that the sampled ones are the
    smallest of all."""
    rng = np.random.default_rng(seed)
    idx = rng.permutation(n).astype(np.int64)
    vals = {"distinct": lambda: 1.0 + rng.permutation(n),
            "few": lambda: 1.0 + rng.integers(0, 3, n),
            "equal": lambda: np.full(n, 2.5)}[kind]()
    at = idx[sampled(n)]
    vals[at] = -1.0 - rng.permutation(SAMPLE) if kind == "distinct" else -1.0
    return idx, vals


def test_sampled_positions_are_one_a_part():
    for n in (SAMPLE, SAMPLE + 1, 1_000_003):
        p = sampled(n)
        first = np.arange(SAMPLE) * n // SAMPLE
        after = (np.arange(SAMPLE) + 1) * n // SAMPLE
        assert (p >= first).all() and (p < after).all()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["distinct", "few", "equal"])
@pytest.mark.parametrize("n", [17_000, 131_072, 131_073, 1_000_003, 5_000_001])
def test_rank_outside_the_bracket(n, kind):
    idx, vals = inputs(n, kind, n)
    order = np.lexsort((np.arange(n), vals))
    rank = np.empty(n, np.int64)
    rank[order] = np.arange(n)
    # ranks above the sampled values, up to the one where the bracket opens
    for goal in (SAMPLE + 100, n // 2, 9 * n // 10):
        got = K.quickstat_index(idx, goal, vals)
        r = rank[idx]
        want = np.concatenate([idx[r < goal], order[goal:goal + 1], idx[r > goal]])
        np.testing.assert_array_equal(got, want)


@pytest.mark.gpu
def test_index_out_of_range_is_refused():
    idx, vals = inputs(100_000, "distinct", 1)
    for where in (0, int(sampled(100_000)[5]), 99_999):
        for wrong in (-1, 100_000):
            bad = idx.copy()
            bad[where] = wrong
            with pytest.raises(_lib.KdError):
                K.quickstat_index(bad, 50_000, vals)
