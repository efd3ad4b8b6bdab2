"""Several PME terms on one context: each term's tables follow its own grid,
order and alpha, whichever terms ran before it.  A term on a shared context
gives the bits that it gives on a context of its own."""
import numpy as np
import pytest

from protomol_amd import water

pytestmark = pytest.mark.gpu
PME = "Coulomb -algorithm PMEwald -reciprocal -correction -interpolation BSpline"


def term(grid=24, order=4, accuracy=1e-6):
    return [grid, grid, grid, 8.0, order, accuracy, -1.0]


def context(make, s, precision):
    c = make(precision)
    c.set_topology(s)
    c.set_boundary(s.box, s.origin, 4.0)
    return c


@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("other", [term(order=6), term(accuracy=1e-4), term(grid=30), term(grid=20, order=6)])
def test_terms_in_turn(gpu_ctx_factory, precision, other):
    print("case: pme terms in turn", precision, other, flush=True)
    s = water.named("water648", seed=5, jitter=0.3)
    v = np.random.default_rng(1).standard_normal((s.n, 3))
    values = [term(), other]

    def results(c, h):
        f, e = c.evaluate([h], s.pos)
        return f, e, c.hessian_vec([h], s.pos, v), c.param_gradients([h], s.pos, lj=False)[0]

    own = []
    for t in values:
        c = context(gpu_ctx_factory, s, precision)
        own.append(results(c, c.force(PME, t)))
    c = context(gpu_ctx_factory, s, precision)
    hs = [c.force(PME, t) for t in values]
    for k in (0, 1, 0, 1):
        for got, want in zip(results(c, hs[k]), own[k]):
            np.testing.assert_array_equal(got, want)
