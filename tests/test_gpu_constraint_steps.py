"""Constrained MD steps whose displacement test and binning run in one launch
after SHAKE (or, with RATTLE alone, in the drift): with reused lists (and,
leapfrog, captured steps) against runs that build their lists on every step,
where that launch only bins, and against steps driven from the host, one
evaluation and one SHAKE or RATTLE call after the other, which have no such
launch.  FP64, 8,100 water atoms, 30 steps; the runs sum the same pairs in
another order (FP64 round-off and the forces' 2^-40 resolution, amplified over
30 steps: 1e-8 A)."""
import numpy as np
import pytest

from protomol_amd import water
from tests.cases import gpu_forces_c1

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("integrator", ["leapfrog", "langevin"])
@pytest.mark.parametrize("shake,rattle", [(True, False), (False, True), (True, True)])
def test_reused_lists_match_fresh_ones(gpu_ctx_factory, integrator, shake, rattle):
    print("case: constrained steps", integrator, shake, rattle, flush=True)
    s = water.named("water8k", seed=6, jitter=0.2)
    got = []
    for fresh in (False, True):
        c = gpu_ctx_factory("double")
        c.set_topology(s)
        c.set_boundary(s.box, s.origin, 4.0)
        if fresh:
            c.set_option("list_skin", 0)
            c.set_option("graph", 0)
        hs = gpu_forces_c1(c)
        kw = dict(temperature=300.0, gamma=5.0, seed=3) if integrator == "langevin" else {}
        c.md_setup(hs, integrator, dt=1.0, **kw)
        c.md_set_state(s.pos, s.vel)
        c.md_set_constraints(1e-10 if shake else 0.0, 100 if shake else 0, 1e-10 if rattle else 0.0, 100 if rattle else 0)
        c.md_run(30)
        got.append(c.md_get_state())
        got[-1] += (c.stats()["list_builds"],)
    (x, v, e, builds), (x0, v0, e0, _) = got
    print("list builds", builds, "max |dx|", np.abs(x - x0).max(), flush=True)
    assert builds < 30
    np.testing.assert_allclose(x, x0, rtol=0, atol=1e-8)
    np.testing.assert_allclose(v, v0, rtol=0, atol=1e-7 * np.abs(v0).max())
    np.testing.assert_allclose(e, e0, rtol=1e-8, atol=1e-8 * np.abs(e0).max())


@pytest.mark.parametrize("shake,rattle", [(True, False), (False, True), (True, True)])
def test_steps_match_host_driven_ones(gpu_ctx_factory, shake, rattle):
    print("case: constrained steps from the host", shake, rattle, flush=True)
    s = water.named("water8k", seed=6, jitter=0.2)
    c = gpu_ctx_factory("double")
    c.set_topology(s)
    c.set_boundary(s.box, s.origin, 4.0)
    hs = gpu_forces_c1(c)
    c.md_setup(hs, "leapfrog", dt=1.0)
    c.md_set_state(s.pos, s.vel)
    c.md_set_constraints(1e-10 if shake else 0.0, 100 if shake else 0, 1e-10 if rattle else 0.0, 100 if rattle else 0)
    c.md_run(30)
    xg, vg, _ = c.md_get_state()
    assert c.stats()["list_builds"] < 30
    h = gpu_ctx_factory("double")
    h.set_topology(s)
    h.set_boundary(s.box, s.origin, 4.0)
    hh = gpu_forces_c1(h)
    x, v = s.pos.copy(), s.vel.copy()
    dt = water.INV_TIMEFACTOR

    def kick(f, part):
        return v + part * dt * f / s.mass[:, None]

    def drift():
        new = x + dt * v
        return h.shake(new, v, x, 1.0, 1e-10, 100)[:2] if shake else (new, v)

    for step in range(31):
        f = h.evaluate(hh, x)[0]
        if 0 < step < 30 and not rattle:
            v = kick(f, 1.0)
        elif step > 0:
            v = kick(f, 0.5)
            if rattle:
                v = h.rattle(x, v, 1.0, 1e-10, 100)[0]
            if step < 30:
                v = kick(f, 0.5)
        else:
            v = kick(f, 0.5)
        if step < 30:
            x, v = drift()
    print("max |dx|", np.abs(xg - x).max(), flush=True)
    np.testing.assert_allclose(xg, x, rtol=0, atol=1e-8)
    np.testing.assert_allclose(vg, v, rtol=0, atol=1e-7 * np.abs(v).max())
