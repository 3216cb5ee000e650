"""The reverse walk's forms: one wavefront for 64 bodies or a workgroup of up
to 16 (the sizes on either side of each change, and trees too shallow for
it), leaf batches of every remainder, and several steps on one tape, against
the oracle's FP64 gradient."""
import numpy as np
import pytest
import torch

import oracle
from multilanguagekdtree_amd import kdtree as K
from multilanguagekdtree_amd.autograd import Adjoint

pytestmark = pytest.mark.gpu

# FP64 sums of the same terms in another order; the ring's star cancels terms
# some 1e3 times larger than their sum
TOL = 1e-11


@pytest.mark.parametrize("n,leaf", [(3, 7), (9, 7), (29, 7), (113, 7), (300, 32), (700, 3),
                                    (16384, 7), (16385, 7), (65536, 8), (65537, 7)])
def test_gradient_matches_oracle(n, leaf):
    b = K.ring(n, seed=n)
    steps = 3 if n < 10000 else 1
    x = np.stack([b[f] for f in "xyz"], 1)
    v = np.stack([b["v" + f] for f in "xyz"], 1)
    rng = np.random.default_rng(n)
    gp, gv = rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    _, tape = oracle.adj_forward(b, 1e-3, steps, 0.3, leaf=leaf)
    ref = oracle.adj_backward(tape, gp, gv)
    sim = Adjoint(n, steps, 2, leaf_size=leaf, precision=K.KD_PREC_FP64)
    t = [torch.as_tensor(a, device="cuda") for a in (x, v, b["m"], gp, gv)]
    sim.forward(*t[:3])
    got = sim.backward(*t[3:])
    sim.close()
    for g, r in zip(got, ref):
        assert np.linalg.norm(g.cpu().numpy() - r) <= TOL * np.linalg.norm(r)
