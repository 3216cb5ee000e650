"""Equal coordinates in a dimension that the build skips at the device-wide
levels and orders per segment: layers of a thin system, which the segments
split (runs of equal keys across medians) or do not.  Trees against the
oracle's, bit for bit, after an upload and from tree order, and what the runs
cost."""
import time

import numpy as np
import pytest

from helpers import compare_trees, pscale
from multilanguagekdtree_amd import kdtree as K

pytestmark = pytest.mark.gpu


def layers(n, thin, layers, gap, seed, jitter=0.0):
    rng = np.random.default_rng(seed)
    p = rng.random((3, n))
    p[thin] = gap * (rng.integers(0, layers, n) + jitter * rng.random(n))
    return dict(zip(K.FIELDS, (*p, *np.zeros((3, n)), rng.uniform(0.5, 1.5, n) / n)))


@pytest.mark.parametrize("thin", [0, 1, 2])
@pytest.mark.parametrize("n,count,gap", [(6000, 4, 1e-2), (6000, 2, 1e-6), (6000, 40, 1e-3),
                                         (50_000, 4, 1e-2), (300_001, 3, 5e-3)])
def test_trees_match_oracle(orc, n, thin, count, gap):
    b = layers(n, thin, count, gap, n + thin)
    r = orc.build_tree(b)
    with K.Simulation(n) as s:
        for _ in range(2):  # the second upload's first build skips a dimension
            s.upload(b)
            for _ in range(2):
                s.build()
                compare_trees(s.export_tree(K.KD_LAYOUT_COMPACT), r, pscale(b))
        assert s.get_tuning("lazy_builds") > 0


def test_runs_do_not_dominate_the_build():
    # four layers, and the same system with no two bodies at one height; runs
    # in any order made this 5.7 ms against 0.8
    n = 1_000_000

    def first_build(b):
        best = float("inf")
        with K.Simulation(n, precision=K.KD_PREC_MIXED) as s:
            for _ in range(6):
                s.upload(b)
                t = time.perf_counter()
                s.build()
                best = min(best, time.perf_counter() - t)
            assert s.get_tuning("lazy_builds") > 0
            times = []
            for _ in range(6):
                t = time.perf_counter()
                s.build()
                times.append(time.perf_counter() - t)
        return best, min(times)

    tied, distinct = (first_build(layers(n, 2, 4, 1e-2, 1, jitter)) for jitter in (0.0, 1e-3))
    assert tied[0] <= 3.0 * distinct[0] and tied[1] <= 3.0 * distinct[1]
