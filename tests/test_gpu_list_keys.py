"""Kept pair lists belong to the pair cutoff that they were built for: force
evaluations of different cutoffs in turn on one context, at positions that
would keep any of the lists, against contexts of their own, and MD runs with
such evaluations between them.  FP64: round-off of sums in another order
(1e-11; 1e-8 A after 20 steps)."""
import numpy as np
import pytest

from protomol_amd import gpu, water
from tests.cases import gpu_forces_c1, rms_rel

pytestmark = pytest.mark.gpu
LJ = "LennardJones CoulombEwaldReal -algorithm NonbondedCutoff -switchingFunction C2 -switchingFunction Cutoff"


def values(rc):
    return [rc - 1.0, rc, 0.4, rc, rc]


def context(make, s, precision, **options):
    c = make(precision)
    c.set_topology(s)
    c.set_boundary(s.box, s.origin, 4.0)
    for k, v in options.items():
        c.set_option(k, v)
    return c


@pytest.mark.parametrize("precision,tol", [("mixed", 5e-6), ("double", 1e-11)])
@pytest.mark.parametrize("options", [{}, {"pair_lanes": 0}, {"prune_skin": 300}, {"cluster_size": 4}])
@pytest.mark.parametrize("cutoffs", [(8.0, 5.0), (5.0, 8.0), (8.0, 9.0, 6.0)])
def test_cutoffs_in_turn(gpu_ctx_factory, precision, tol, options, cutoffs):
    print("case: list cutoffs in turn", precision, options, cutoffs, flush=True)
    s = water.named("water648", seed=5, jitter=0.3)
    own = []
    for rc in cutoffs:
        c = context(gpu_ctx_factory, s, precision, **options)
        own.append(c.evaluate([c.force(LJ, values(rc))], s.pos))
    c = context(gpu_ctx_factory, s, precision, **options)
    hs = [c.force(LJ, values(rc)) for rc in cutoffs]
    for k in list(range(len(cutoffs))) * 2:
        f, e = c.evaluate([hs[k]], s.pos + 0.01)     # (all atoms alike: the same forces)
        assert rms_rel(f, own[k][0]) < tol
        np.testing.assert_allclose(e[:2], own[k][1][:2], rtol=10 * tol)


@pytest.mark.parametrize("integrator", ["leapfrog", "langevin"])
@pytest.mark.parametrize("other", [5.0, 9.0])
def test_md_after_another_cutoff(gpu_ctx_factory, integrator, other):
    print("case: md after another cutoff", integrator, other, flush=True)
    s = water.named("water648", seed=6, jitter=0.2)
    got = []
    for between in (True, False):
        c = context(gpu_ctx_factory, s, "double")
        hs = [c.force(LJ, values(8.0)), c.force("Bond", []), c.force("Angle", [])]
        o = c.force(LJ, values(other))
        kw = dict(temperature=300.0, gamma=5.0, seed=3) if integrator == "langevin" else {}
        c.md_setup(hs, integrator, dt=1.0, **kw)
        c.md_set_state(s.pos, s.vel)
        for _ in range(3):
            c.md_run(20)
            x, v, _ = c.md_get_state()
            if between:
                c.evaluate([o], x)
            else:
                c.md_set_state(x, v)
        got.append(c.md_get_state()[:2])
    np.testing.assert_allclose(got[0][0], got[1][0], rtol=0, atol=1e-7)
    np.testing.assert_allclose(got[0][1], got[1][1], rtol=0, atol=1e-6 * np.abs(got[1][1]).max())


# a group whose last pass has the smaller cutoff: the lists have room for the
# widest pass (each pass is rounded to 2^-40 on its own, so the sums agree)
@pytest.mark.parametrize("precision", ["mixed", "double"])
@pytest.mark.parametrize("order", [(0, 1), (1, 0)])
def test_capacity_of_the_widest_pass(gpu_ctx_factory, precision, order):
    print("case: list capacity over passes", precision, order, flush=True)
    s = water.named("water8k", seed=5, jitter=0.3)
    c = context(gpu_ctx_factory, s, precision, list_skin=0)
    hs = [c.force("LennardJones -algorithm NonbondedCutoff -switchingFunction C2", [11.0, 12.0, 12.0]),
          c.force("Coulomb -algorithm NonbondedCutoff -switchingFunction C2", [3.0, 4.0, 4.0])]
    parts = [c.evaluate([h], s.pos) for h in hs]
    f, e = c.evaluate([hs[k] for k in order], s.pos)
    want = parts[0][0] + parts[1][0]
    assert np.abs(f - want).max() <= 4 * 2.0 ** -40 + 1e-14 * np.abs(want).max()
    np.testing.assert_allclose(e, parts[0][1] + parts[1][1], rtol=1e-12, atol=1e-9)
    v = np.random.default_rng(3).standard_normal((s.n, 3))
    want = c.hessian_vec(hs[:1], s.pos, v) + c.hessian_vec(hs[1:], s.pos, v)
    assert np.abs(c.hessian_vec([hs[k] for k in order], s.pos, v) - want).max() <= 1e-10 * np.abs(want).max()


# the lists of a run that replicas repeat are in their own order whatever the
# context evaluated before the run was set up: the same bits
@pytest.mark.parametrize("before", ["evaluate", "leapfrog"])
def test_replica_run_after_other_work(gpu_ctx_factory, before):
    print("case: replica run after", before, flush=True)
    s = water.water_box(300, (300 / 0.0334) ** (1.0 / 3.0), seed=8, jitter=0.2)
    got = []
    for prepare in (True, False):
        c = context(gpu_ctx_factory, s, "mixed")
        hs = gpu_forces_c1(c) + [c.force("Bond", []), c.force("Angle", [])]
        if prepare and before == "evaluate":
            c.evaluate(hs, s.pos)
        elif prepare:
            c.md_setup(hs, "leapfrog", dt=1.0)
            c.md_set_state(s.pos, s.vel)
            c.md_run(1)
        c.md_setup(hs, "langevin", dt=1.0, temperature=400.0, gamma=5.0, seed=3)
        c.md_set_state(s.pos, s.vel)
        c.md_run(30)
        got.append(c.md_get_state())
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


# cell diagnostics between two runs replace positions and cell lists: the next
# run starts from their positions with forces and lists of its own
@pytest.mark.parametrize("integrator", ["leapfrog", "langevin"])
def test_md_after_cell_diagnostics(gpu_ctx_factory, integrator):
    print("case: md after cell diagnostics", integrator, flush=True)
    s = water.named("water648", seed=7, jitter=0.2)
    move = np.repeat(np.random.default_rng(5).uniform(-0.15, 0.15, (s.n // 3, 3)), 3, axis=0)
    got = []
    for diagnostics in (True, False):
        c = context(gpu_ctx_factory, s, "double")
        hs = [c.force(LJ, values(8.0)), c.force("Bond", []), c.force("Angle", []),
              c.force("Coulomb -algorithm PMEwald -reciprocal -correction -interpolation BSpline",
                      [24, 24, 24, 8.0, 4, 1e-6, 0.4])]
        kw = dict(temperature=300.0, gamma=5.0, seed=3) if integrator == "langevin" else {}
        c.md_setup(hs, integrator, dt=0.5, **kw)
        c.md_set_state(s.pos, s.vel)
        for _ in range(3):
            c.md_run(20)
            x, v, _ = c.md_get_state()
            if diagnostics:
                c.cell_diagnostics(x + move, 8.0, 8.0)
            else:
                c.md_set_state(x + move, v)
        c.md_run(20)
        got.append(c.md_get_state()[:2])
    np.testing.assert_allclose(got[0][0], got[1][0], rtol=0, atol=1e-7)
    np.testing.assert_allclose(got[0][1], got[1][1], rtol=0, atol=1e-6 * np.abs(got[1][1]).max())


def test_refused_cutoff_between(gpu_ctx_factory):
    """A cutoff whose cell stencil is too large is refused before anything is
    allocated or queued, and the lists around it still hold."""
    print("case: refused cutoff between", flush=True)
    s = water.named("water8k", seed=5, jitter=0.3)
    c = gpu_ctx_factory("double")
    c.set_topology(s)
    c.set_boundary(s.box, s.origin, 1.2)
    h, wide = c.force(LJ, values(8.0)), c.force(LJ, values(30.0))
    want = c.evaluate([h], s.pos)
    builds = c.stats()["list_builds"]
    for _ in range(2):
        with pytest.raises(gpu.PmError) as e:
            c.evaluate([wide], s.pos)
        assert e.value.code == gpu.PM_ERR_UNSUPPORTED
        got = c.evaluate([h], s.pos)
        np.testing.assert_array_equal(got[0], want[0])
        np.testing.assert_array_equal(got[1], want[1])
    assert c.stats()["list_builds"] == builds
