"""FP64 gradients of systems with bodies so far apart that powers of their
distances overflow (its cube above 2e102, its square above 1e154): such pairs
add nothing, the others keep their terms.  Against the oracle's gradient."""
import numpy as np
import pytest

import oracle
from multilanguagekdtree_amd import kdtree as K

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from multilanguagekdtree_amd.autograd import Adjoint  # noqa: E402

TOL = 1e-11  # FP64 sums of the same terms in another order


@pytest.mark.parametrize("far", [1e60, 1e95, 1e110, 1e150, 3e154])
@pytest.mark.parametrize("n", [40, 1000])
def test_bodies_far_apart(n, far):
    rng = np.random.default_rng(n)
    p = rng.normal(size=(n, 3))
    p[:8] = far * (1.0 + np.arange(24).reshape(8, 3))  # every difference is as large
    v = 0.1 * rng.normal(size=(n, 3))
    m = rng.uniform(0.5, 1.5, n) / n
    b = dict(zip(K.FIELDS, (*np.ascontiguousarray(p.T), *np.ascontiguousarray(v.T), m)))
    gp, gv = rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    steps = 2
    _, tape = oracle.adj_forward(b, 1e-3, steps, 0.3)
    ref = oracle.adj_backward(tape, gp, gv)
    sim = Adjoint(n, steps, 2, precision=K.KD_PREC_FP64)
    t = [torch.as_tensor(np.ascontiguousarray(a), device="cuda") for a in (p, v, m, gp, gv)]
    sim.forward(*t[:3])
    got = sim.backward(*t[3:])
    sim.close()
    for g, r in zip(got, ref):
        g = g.cpu().numpy()
        assert np.isfinite(r).all() and np.isfinite(g).all()
        assert np.linalg.norm(g - r) <= TOL * np.linalg.norm(r)
