"""SHAKE and RATTLE around the constraint kernels' launch limits: sweep counts
at and beside those the first probe records (16), and group counts on both
sides of one-wave and four-wave blocks (65,536 groups), bit for bit against
the oracle (the same FP64 operations in the same order)."""
import numpy as np
import pytest

from protomol_amd import water

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("molecules", [1, 65, 217])
@pytest.mark.parametrize("eps,max_iter", [(1e-300, 1), (1e-300, 15), (1e-300, 16), (1e-300, 17), (1e-300, 21), (1e-5, 16), (1e-5, 30), (1e-9, 40)])
def test_sweep_counts(gpu_ctx_factory, port, molecules, eps, max_iter):
    check(gpu_ctx_factory, port, molecules, eps, max_iter)


@pytest.mark.parametrize("molecules", [65536, 65537])
def test_block_sizes(gpu_ctx_factory, port, molecules):
    check(gpu_ctx_factory, port, molecules, 1e-9, 30)


def check(make, port, molecules, eps, max_iter):
    print("case: constraint probe", molecules, eps, max_iter, flush=True)
    s = water.water_box(molecules, max(10.0, (molecules / 0.0334) ** (1.0 / 3.0)), seed=molecules)
    rng = np.random.default_rng(molecules)
    x = s.pos + 0.03 * rng.standard_normal(s.pos.shape)
    c = make("double")
    c.set_topology(s)
    c.set_boundary(s.box, s.origin, 4.0)
    cons = port.constraint_list(s)
    xg, vg, kg = c.shake(x, s.vel, s.pos, 1.0, eps, max_iter)
    xo, vo, _, ko = port.shake(cons, s.mass, x, s.vel, s.pos, 1.0, eps, max_iter)
    assert kg == ko
    np.testing.assert_array_equal(xg, xo)
    np.testing.assert_array_equal(vg, vo)
    vg, kg = c.rattle(xo, s.vel, 1.0, eps, max_iter)
    vo, ko = port.rattle(cons, s.mass, xo, s.vel, 1.0, eps, max_iter)
    assert kg == ko
    np.testing.assert_array_equal(vg, vo)
