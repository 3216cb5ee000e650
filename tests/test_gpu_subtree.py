"""The subtree builder's forms: a system of one segment, which sorts every
dimension itself, grids on either side of one workgroup a CU (where a
segment's coordinates stay in LDS), and leaf sizes whose node sums do and do
not fit beside the staged terms.  Trees against the oracle's, bit for bit,
from the upload's order and from tree order."""
import numpy as np
import pytest

from helpers import compare_trees, pscale
from multilanguagekdtree_amd import kdtree as K

pytestmark = pytest.mark.gpu


def cloud(n, seed):
    # equal coordinates, and values closer together than the sorts' keys
    rng = np.random.default_rng(seed)
    p = rng.normal(size=(3, n))
    near = rng.random(n) < 0.3
    p[:, near] = 1.0 + rng.uniform(0.0, 2.0 ** -24, (3, int(near.sum())))
    same = rng.random(n) < 0.1
    p[1, same] = 0.5
    return dict(zip(K.FIELDS, (*p, *np.zeros((3, n)), rng.uniform(0.5, 2.0, n) / n)))


@pytest.mark.parametrize("n,leaf", [(2, 2), (65, 2), (513, 7), (1221, 7), (1793, 7), (2048, 2),
                                    (2048, 32), (2049, 7), (300_000, 7), (524_288, 7),
                                    (524_289, 32)])
def test_trees_match_oracle(orc, n, leaf):
    b = cloud(n, n)
    r = orc.build_tree(b, leaf)
    with K.Simulation(n, leaf_size=leaf) as s:
        s.upload(b)
        for _ in range(2):
            s.build()
            compare_trees(s.export_tree(K.KD_LAYOUT_COMPACT), r, pscale(b))
