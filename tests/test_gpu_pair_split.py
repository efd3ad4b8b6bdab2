"""Where the lane-per-entry pair kernel's launch changes (waves per cluster,
waves per block) and where its list groups and skipped terms can go wrong:
forces and energies against the oracle, at fresh positions and, with the kept
lists, after moves that bring far entries within the cutoff.  Tolerances: the
mixed-precision force bar (5e-6 RMS relative, FP32 pair arithmetic) and FP64
round-off of sums of ~300 terms (1e-11)."""
import numpy as np
import pytest

from oracle import pyoracle as po
from protomol_amd import water
from tests.cases import exclusion_mix, gpu_forces_c1, rms_rel

pytestmark = pytest.mark.gpu
TOL = {"mixed": 5e-6, "double": 1e-11}


def reference(port, s, x):
    t = s.copy()
    t.pos = x
    a = port.cutoff(t, [po.term(po.POT_LJ, po.SWF_C2, 8.0, 7.0)], 8.0, 4.0)
    b = port.cutoff(t, [po.term(po.POT_COULOMB, po.SWF_C2, 8.0, 7.0)], 8.0, 4.0)
    return a["forces"] + b["forces"], a["energies"] + b["energies"]


# molecules: 8 (two sizes), 4, 2 and 1 (two sizes) waves per cluster, as many
# as keep the launch within 1,024 waves
@pytest.mark.parametrize("molecules", [150, 217, 300, 600, 1301, 2600])
@pytest.mark.parametrize("kind", ["water", "exclusions", "uncharged"])
@pytest.mark.parametrize("precision", ["mixed", "double"])
def test_pair_forces_over_launch_shapes(gpu_ctx_factory, port, molecules, kind, precision):
    print("case: pair split", molecules, kind, precision, flush=True)
    s = water.water_box(molecules, (molecules / 0.0334) ** (1.0 / 3.0), seed=molecules, jitter=0.3)
    if kind == "exclusions":
        s = exclusion_mix(s)          # hydrogens with Lennard-Jones, 1-4 pairs
    if kind == "uncharged":
        s.q = np.where(np.arange(s.n) % 7 == 3, 0.0, s.q)
    c = gpu_ctx_factory(precision)
    c.set_topology(s)
    c.set_boundary(s.box, s.origin, 4.0)
    hs = gpu_forces_c1(c)
    rng = np.random.default_rng(molecules)
    builds = None
    # the second move keeps the lists (half the skin is 1.1 A mixed, 0.5 FP64)
    # and carries pairs from outside the near margin (0.5 A) into the cutoff
    for step in (0.0, 0.45):
        d = rng.standard_normal((molecules, 3))
        x = s.pos + step * np.repeat(d / np.linalg.norm(d, axis=1)[:, None], 3, axis=0)
        f, e = c.evaluate(hs, x)
        if builds is not None:
            assert c.stats()["list_builds"] == builds
        builds = c.stats()["list_builds"]
        fr, er = reference(port, s, x)
        err = rms_rel(f, fr)
        print("rms rel force", err, flush=True)
        assert err < TOL[precision]
        np.testing.assert_allclose(e[:2], er[:2], rtol=10 * TOL[precision], atol=1e-6 * np.abs(er[:2]).max())


# blocks of 8 waves beside PME in mixed precision up to 163,840 slots: 163,688
# and 163,992, beside PME and alone, against the row-per-entry kernel
# (5e-6: FP32 pair arithmetic on both sides)
@pytest.mark.parametrize("molecules", [52600, 52700])
def test_forces_over_block_widths(gpu_ctx_factory, molecules):
    print("case: block widths", molecules, flush=True)
    s = water.water_box(molecules, (molecules / 0.0334) ** (1.0 / 3.0), seed=molecules, jitter=0.3)
    got = []
    for lanes in (0, 1):
        c = gpu_ctx_factory("mixed")
        c.set_topology(s)
        c.set_boundary(s.box, s.origin, 4.0)
        c.set_option("pair_lanes", lanes)
        hs = gpu_forces_c1(c)
        pme = c.force("Coulomb -algorithm PMEwald -reciprocal -correction -interpolation BSpline",
                      [108, 108, 108, 8.0, 4, 1e-6, -1.0])
        alone, both = c.evaluate(hs, s.pos), c.evaluate(hs + [pme], s.pos)
        p = c.evaluate([pme], s.pos)
        got.append((alone, (both[0] - p[0], both[1] - p[1])))
    for (f, e), (fr, er) in zip(got[1], got[0]):
        assert rms_rel(f, fr) < TOL["mixed"]
        np.testing.assert_allclose(e[:2], er[:2], rtol=1e-4)


# the scan of up to 16,384 atoms (3,072 where every evaluation builds its
# lists) also scatters them: a box on each side
@pytest.mark.parametrize("molecules,skin", [(5461, -1), (5462, -1), (1024, 0), (1025, 0)])
def test_forces_over_layout_launches(gpu_ctx_factory, port, molecules, skin):
    print("case: layout launches", molecules, skin, flush=True)
    s = water.water_box(molecules, (molecules / 0.0334) ** (1.0 / 3.0), seed=molecules, jitter=0.3)
    c = gpu_ctx_factory("double")
    c.set_topology(s)
    c.set_boundary(s.box, s.origin, 4.0)
    c.set_option("list_skin", skin)
    f, _ = c.evaluate(gpu_forces_c1(c), s.pos)
    assert rms_rel(f, reference(port, s, s.pos)[0]) < TOL["double"]
