"""Forces of the second stream (PME, correction) beside the bonded terms of
the first: every combination of a reciprocal term, a second one and a
correction without one gives the sum of its parts.  Each part is rounded to
2^-40 kcal/mol/A per atom and term on its own, so the sums agree to a few
such units."""
import numpy as np
import pytest

from protomol_amd import water

pytestmark = pytest.mark.gpu
PME = "Coulomb -algorithm PMEwald %s -interpolation BSpline"


@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("parts", [("recip", "bond"), ("corr", "bond"), ("recip", "both"), ("corr", "recip", "angle"),
                                   ("both", "pair", "bond", "angle"), ("corr", "pair", "angle")])
def test_side_forces_add_up(gpu_ctx_factory, precision, parts):
    print("case: side forces", precision, parts, flush=True)
    s = water.named("water648", seed=5, jitter=0.3)
    s.pos = s.pos + np.random.default_rng(6).normal(0.0, 0.03, s.pos.shape)
    c = gpu_ctx_factory(precision)
    c.set_topology(s)
    c.set_boundary(s.box, s.origin, 4.0)
    v = [24, 24, 24, 8.0, 4, 1e-6, -1.0]
    make = {"recip": lambda: c.force(PME % "-reciprocal", v), "corr": lambda: c.force(PME % "-correction", v),
            "both": lambda: c.force(PME % "-reciprocal -correction", v), "bond": lambda: c.force("Bond", []),
            "angle": lambda: c.force("Angle", []),
            "pair": lambda: c.force("LennardJones -algorithm NonbondedCutoff -switchingFunction C2", [7.0, 8.0, 8.0])}
    hs = [make[p]() for p in parts]
    single = [c.evaluate([h], s.pos) for h in hs]
    for _ in range(2):      # the second call finds the buffers of the first
        f, e = c.evaluate(hs, s.pos)
        want = sum(x[0] for x in single)
        assert np.abs(f - want).max() <= 16 * 2.0 ** -40 + 1e-15 * np.abs(want).max()
        np.testing.assert_allclose(e, sum(x[1] for x in single), rtol=1e-12, atol=1e-9)
