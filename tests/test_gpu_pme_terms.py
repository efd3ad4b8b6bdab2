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


# two reciprocal terms in one group, the smaller grid first and last, and the
# same term twice: each part is computed on its own in either case, so the sum
# of the parts agrees to FP64 round-off of the sums (and, forces, to the 2^-40
# steps that the parts are rounded to)
@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("spread", [1, 0])
@pytest.mark.parametrize("values", [[term(), term(grid=32, order=6)], [term(grid=32, order=6), term()],
                                    [term(), term(accuracy=1e-4)], [term(), term()],
                                    [term(), term(grid=20), term(grid=30), term(order=6), term(grid=32, order=8)]])
def test_terms_of_a_group_add_up(gpu_ctx_factory, precision, spread, values):
    print("case: pme terms of a group", precision, spread, values, flush=True)
    s = water.named("water648", seed=6, jitter=0.3)
    v = np.random.default_rng(2).standard_normal((s.n, 3))
    c = context(gpu_ctx_factory, s, precision)
    c.set_option("pme_spread", spread)
    hs = [c.force(PME, t) for t in values]
    for _ in range(2):
        f, e = c.evaluate(hs, s.pos, virial=True)
        hv = c.hessian_vec(hs, s.pos, v)
        dq = c.param_gradients(hs, s.pos, lj=False)[0]
        vals, _, _, alpha, beta = c.lanczos(hs, s.pos, v, steps=3)
        parts = [c.evaluate([h], s.pos, virial=True) for h in hs]
        want = sum(p[0] for p in parts)
        assert np.abs(f - want).max() <= 16 * 2.0 ** -40 + 1e-14 * np.abs(want).max()
        np.testing.assert_allclose(e, sum(p[1] for p in parts), rtol=1e-12, atol=1e-9)
        want = sum(c.hessian_vec([h], s.pos, v) for h in hs)
        assert np.abs(hv - want).max() <= 1e-12 * np.abs(want).max()
        want = sum(c.param_gradients([h], s.pos, lj=False)[0] for h in hs)
        assert np.abs(dq - want).max() <= 1e-12 * np.abs(want).max()
        # the Lanczos recurrence over single products
        V, ra, rb = [v.reshape(-1) / np.linalg.norm(v)], [], []
        for _ in range(3):
            w = c.hessian_vec(hs, s.pos, V[-1].reshape(-1, 3)).reshape(-1)
            ra.append(V[-1] @ w)
            for _ in range(2):
                for u in V:
                    w = w - (u @ w) * u
            rb.append(np.linalg.norm(w))
            V.append(w / rb[-1])
        # (the directions agree to FP64 round-off; their FP32 copies in mixed
        # precision to 6e-8, which three steps amplify by a few tens)
        tol = (1e-5 if precision == "mixed" else 1e-11) * max(np.abs(ra).max(), np.abs(rb).max())
        np.testing.assert_allclose(alpha, ra, rtol=0, atol=tol)
        np.testing.assert_allclose(beta, rb, rtol=0, atol=tol)


# two real terms in a box no wider than twice their cutoffs, each with the
# lattice images of its own cutoff
@pytest.mark.parametrize("cutoffs", [(14.0, 9.4), (9.4, 14.0)])
def test_real_terms_of_two_cutoffs(gpu_ctx_factory, cutoffs):
    print("case: real terms of two cutoffs", cutoffs, flush=True)
    s = water.named("water648", seed=8, jitter=0.3)
    c = context(gpu_ctx_factory, s, "double")
    hs = [c.force("Coulomb -algorithm PMEwald -real -correction -interpolation BSpline", [24, 24, 24, rc, 4, 1e-6, 0.15])
          for rc in cutoffs]
    f, e = c.evaluate(hs, s.pos)
    parts = [c.evaluate([h], s.pos) for h in hs]
    want = parts[0][0] + parts[1][0]
    assert np.abs(f - want).max() <= 16 * 2.0 ** -40 + 1e-14 * np.abs(want).max()
    np.testing.assert_allclose(e, parts[0][1] + parts[1][1], rtol=1e-12, atol=1e-9)


# tables of a large grid (theta over 64 MB) go back when another term needs
# its own, and are filled again
def test_large_grids_in_turn(gpu_ctx_factory):
    print("case: large pme grids in turn", flush=True)
    s = water.named("water648", seed=9, jitter=0.3)
    c = context(gpu_ctx_factory, s, "double")
    hs = [c.force(PME, term(grid=g)) for g in (256, 24, 288)]
    want = [c.evaluate([h], s.pos) for h in hs]
    for k in (0, 2, 1, 2, 0):
        f, e = c.evaluate([hs[k]], s.pos)
        np.testing.assert_array_equal(f, want[k][0])
        np.testing.assert_array_equal(e, want[k][1])
    f, _ = c.evaluate(hs, s.pos)
    total = sum(w[0] for w in want)
    assert np.abs(f - total).max() <= 16 * 2.0 ** -40 + 1e-14 * np.abs(total).max()
