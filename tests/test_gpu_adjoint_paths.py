"""The adjoint's launch variants against each other in FP64: the PME spread of
both grids inside the forward transform (pme_spread 1) and as kernels of their
own (0), one and two pair passes, no PME, the smallest box (16 waves per
cluster) and a larger one; and a Lanczos run, whose later steps keep the
layout, the lists and the charges' potential of the first, against the same
recurrence over single Hessian-vector products.  The variants sum the same
terms in another order: FP64 round-off plus the 2^-40 resolution of the pair
sums, of about 1e3 terms each (1e-9)."""
import numpy as np
import pytest

from protomol_amd import gpu, water
from tests.cases import ALPHA_RC8, rms_rel
from tests.test_gpu_adjoint import away_from_cutoff, unit

pytestmark = pytest.mark.gpu

LJ_COUL = ("LennardJones CoulombEwaldReal -algorithm NonbondedCutoff -switchingFunction C2 -switchingFunction Cutoff",
           [7.0, 8.0, ALPHA_RC8, 8.0, 8.0])
LJ = ("LennardJones -algorithm NonbondedCutoff -switchingFunction C2", [6.0, 7.0, 7.0])
COUL = ("CoulombEwaldReal -algorithm NonbondedCutoff -switchingFunction Cutoff", [ALPHA_RC8, 8.0, 8.0])
FORCES = {"one pass": [LJ_COUL], "two passes": [LJ, COUL]}


def context(make, s, forces, pme, spread=1, sigma=None, eps=None):
    c = make("double")
    c.set_topology(s)
    c.set_boundary(s.box, s.origin, 4.0)
    if sigma is not None:
        c.set_lj_per_atom(sigma, eps)
    c.set_option("pme_spread", spread)
    ids = list(FORCES[forces])
    if pme:
        g = 32 if s.n < 1000 else 48
        ids.append(("Coulomb -algorithm PMEwald -reciprocal -correction -interpolation BSpline",
                    [g, g, g, 8.0, pme, 1e-6, -1.0]))
    return c, [c.force(i, v) for i, v in ids]


@pytest.mark.parametrize("box", ["water648", "water8k"])
@pytest.mark.parametrize("forces", ["one pass", "two passes"])
@pytest.mark.parametrize("order", [4, 6])
def test_spread_variants_agree(gpu_ctx_factory, box, forces, order):
    print("case: adjoint spread variants", box, forces, order, flush=True)
    s, sigma, eps = water.perturbed_box(box, seed=3)
    v = np.random.default_rng(7).standard_normal((s.n, 3))
    got = []
    for spread in (1, 0):
        c, hs = context(gpu_ctx_factory, s, forces, order, spread, sigma, eps)
        got.append([c.hessian_vec(hs, s.pos, v), *c.param_gradients(hs, s.pos)])
    for a, b in zip(*got):
        assert rms_rel(a, b) < 1e-9


@pytest.mark.parametrize("forces", ["one pass", "two passes"])
@pytest.mark.parametrize("pme", [0, 4])
@pytest.mark.parametrize("spread", [1, 0])
def test_lanczos_matches_single_products(gpu_ctx_factory, forces, pme, spread):
    print("case: lanczos against single products", forces, pme, spread, flush=True)
    s = water.named("water648", seed=21, jitter=0.4)
    c, hs = context(gpu_ctx_factory, s, forces, pme, spread)
    m = 6
    v0 = np.random.default_rng(9).standard_normal((s.n, 3))
    c.hessian_vec(hs, s.pos + 0.1, v0)   # another layout and potential before
    _, _, _, alpha, beta = c.lanczos(hs, s.pos, v0, steps=m)
    V = [v0.reshape(-1) / np.linalg.norm(v0)]
    ra, rb = [], []
    for _ in range(m):
        w = c.hessian_vec(hs, s.pos, V[-1].reshape(-1, 3)).reshape(-1)
        ra.append(V[-1] @ w)
        for _ in range(2):
            for u in V:
                w = w - (u @ w) * u
        rb.append(np.linalg.norm(w))
        V.append(w / rb[-1])
    scale = max(np.abs(ra).max(), np.abs(rb).max())
    np.testing.assert_allclose(alpha, ra, rtol=0, atol=1e-8 * scale)
    np.testing.assert_allclose(beta, rb, rtol=0, atol=1e-8 * scale)


def test_refused_parameters_change_nothing(gpu_ctx_factory):
    """A refused pm_set_lj_per_atom leaves a context without per-atom
    parameters without them, and one with them as it was."""
    print("case: refused per-atom parameters", flush=True)
    s, sigma, eps = water.perturbed_box("water648", seed=3)
    bad = sigma.copy()
    bad[5] = -1.0
    c, hs = context(gpu_ctx_factory, s, "one pass", 4)
    with pytest.raises(gpu.PmError):
        c.set_lj_per_atom(bad, eps)
    with pytest.raises(gpu.PmError) as e:
        c.param_gradients(hs, s.pos)
    assert e.value.code == gpu.PM_ERR_STATE
    c.set_lj_per_atom(sigma, eps)
    want = c.param_gradients(hs, s.pos)
    with pytest.raises(gpu.PmError):
        c.set_lj_per_atom(2.0 * bad, 3.0 * eps)
    for a, b in zip(c.param_gradients(hs, s.pos), want):
        np.testing.assert_array_equal(a, b)


# 16, 8, 4, 2 and 1 waves per cluster (as many as keep the launch within
# 16,384): H v against central differences of the forces, h = 1e-4 A (FP64;
# the truncation of second order is 1e-7 of the largest terms, round-off less).
# The second derivative of a C2-switched term jumps at its cutoff: atoms of
# pairs that the differences could carry across it stay put
@pytest.mark.parametrize("molecules", [300, 4000, 9000, 20000, 30000])
def test_products_over_launch_shapes(gpu_ctx_factory, molecules):
    print("case: adjoint launch shapes", molecules, flush=True)
    s = water.water_box(molecules, (molecules / 0.0334) ** (1.0 / 3.0), seed=molecules, jitter=0.3)
    c = gpu_ctx_factory("double")
    c.set_topology(s)
    c.set_boundary(s.box, s.origin, 4.0)
    hs = [c.force(*LJ), c.force("Coulomb -algorithm NonbondedCutoff -switchingFunction C2", [6.0, 7.0, 7.0])]
    v, _ = away_from_cutoff(s, unit(np.random.default_rng(molecules), (s.n, 3)), 7.0)
    h = 1e-4
    fd = -(c.evaluate(hs, s.pos + h * v)[0] - c.evaluate(hs, s.pos - h * v)[0]) / (2 * h)
    assert rms_rel(c.hessian_vec(hs, s.pos, v), fd) < 2e-6
