"""The work that a user of this library has it do, as cases to be timed.

Every case goes through the Python binding of the C ABI (protomol_amd.gpu) as
a program does: force evaluations from host arrays (a SystemForce adapter), MD
runs that start from a host state and hand it back (an output interval of a
simulation), Hessian-vector products, parameter gradients and Lanczos runs (a
normal-mode or parameter-fitting program), and batches of replicas with
exchange.  Systems are three-site water boxes at liquid density (0.0334
molecules per A^3, the size range of protomol_amd/water.py's workloads: 648 to
a million atoms) and the solvated protein of tests/golden/examples/bpti.

exact() restates the whole path in 64 bits with torch alone.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

from protomol_amd import front, gpu, water

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BPTI = os.path.join(ROOT, "tests", "golden", "examples", "bpti")
DENSITY = 0.0334
KB = water.BOLTZMANN
TIME = water.INV_TIMEFACTOR
MD, RIGID, EVAL, HV, PARAM, LANCZOS, REM, PROTEIN = ("md", "rigid", "evaluate", "hessian_vec", "param_gradients",
                                                     "lanczos", "replicas", "protein")


# ------------------------------------------------------------------- cases
def listed():
    return [
        # one force evaluation of a small box, energies included: what a host
        # integrator asks for at every step; the call's latency is its cost
        dict(name="evaluate_648", path=EVAL, molecules=216, precision="mixed", field="cutoff", rc=8.0, grid=0, order=0,
             virial=False),
        # an output interval of a small simulation in the reference's own
        # arithmetic (FP64, plain cutoffs): pmrun's default precision
        dict(name="md_648_double", path=MD, molecules=216, precision="double", field="cutoff", rc=8.0, grid=0, order=0,
             steps=25),
        # a solvated protein (14,281 atoms, every bonded term, scaled 1-4
        # pairs, PME in a box that is not a cube), the reference's PME example
        dict(name="md_protein", path=PROTEIN, precision="mixed", steps=25),
        # second derivatives: one Hessian-vector product (a Newton or
        # normal-mode step) on a mid-sized box with PME
        dict(name="hessian_vec_8k", path=HV, molecules=2700, precision="mixed", field="pme", rc=9.0, grid=48, order=4),
        # gradients with respect to charges and per-atom Lennard-Jones
        # parameters, the backward pass of a parameter fit
        dict(name="param_gradients_8k", path=PARAM, molecules=2700, precision="mixed", field="pme", rc=9.0, grid=48,
             order=4),
        # lowest modes: 30 mass-weighted Lanczos steps with Ritz vectors, FP64
        dict(name="lanczos_8k_double", path=LANCZOS, molecules=2700, precision="double", field="pme", rc=9.0, grid=48,
             order=4, steps=30),
        # the drop-in route at the size of the headline benchmark: host arrays
        # in and out, every energy, in both arithmetics (FP64 with the virial)
        dict(name="evaluate_98k", path=EVAL, molecules=32768, precision="mixed", field="pme", rc=10.0, grid=96, order=4,
             virial=False),
        dict(name="evaluate_98k_double", path=EVAL, molecules=32768, precision="double", field="pme", rc=10.0, grid=96,
             order=4, virial=True),
        # the headline benchmark's system: resident MD with PME
        dict(name="md_98k", path=MD, molecules=32768, precision="mixed", field="pme", rc=10.0, grid=96, order=4, steps=50),
        # the same system with rigid water (SHAKE) at 2 fs
        dict(name="rigid_98k", path=RIGID, molecules=32768, precision="mixed", field="pme", rc=10.0, grid=96, order=4,
             steps=25),
        # the largest: a million atoms
        dict(name="md_1m", path=MD, molecules=333333, precision="mixed", field="pme", rc=10.0, grid=240, order=4, steps=16),
        # replica exchange: 64 boxes of uneven sizes, one exchange interval
        dict(name="replicas_64", path=REM, replicas=64, sizes=0, precision="mixed", steps=50),
    ]


def _grid(edge):
    """The next even size of factors 2, 3 and 5 with at most 1.04 A between grid points."""
    g = max(12, int(math.ceil(edge / 1.04)))
    while True:
        m = g
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1 and g % 2 == 0:
            return g
        g += 1


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _edge(molecules):
    return (molecules / DENSITY) ** (1.0 / 3.0)


def draw(rng):
    path = rng.choice([EVAL, EVAL, EVAL, MD, MD, MD, RIGID, HV, PARAM, LANCZOS, REM, PROTEIN])
    precision = rng.choice(["mixed", "mixed", "double"])
    if path == REM:
        return dict(path=path, replicas=_log(rng, 8, 64), sizes=rng.randint(1, 1000), precision="mixed",
                    steps=rng.randint(10, 50))
    if path == PROTEIN:
        return dict(path=path, precision=precision, steps=rng.randint(5, 40))
    top = {EVAL: 32768, MD: 120000, RIGID: 32768, HV: 11000, PARAM: 11000, LANCZOS: 4000}[path]
    c = dict(path=path, molecules=_log(rng, 216, top), precision=precision)
    edge = _edge(c["molecules"])
    rc = rng.choice([r for r in (8.0, 9.0, 10.0) if 2 * r <= edge])
    pme = rng.random() < 0.7
    c.update(field="pme" if pme else "cutoff", rc=rc, grid=_grid(edge) if pme else 0,
             order=(4 if rng.random() < 0.75 else 6) if pme else 0)
    if path == EVAL:
        c["virial"] = rng.random() < 0.5
    if path in (MD, RIGID):
        c["steps"] = rng.randint(5, 40) if c["molecules"] < 40000 else rng.randint(5, 15)
    if path == LANCZOS:
        c["steps"] = rng.randint(10, 30)
    return c


# ----------------------------------------------------------------- systems
def _boxes(case, seed):
    """The systems of a case (one, or one per replica)."""
    rng = np.random.default_rng([seed, 77])
    if case["path"] == PROTEIN:
        t = front.load_system(os.path.join(BPTI, "bpti.psf"), os.path.join(BPTI, "bpti.par"))
        x = front.read_coords(os.path.join(BPTI, "bpti.pdb"))
        vel = rng.standard_normal(x.shape) * np.sqrt(KB * 300.0 / t.mass)[:, None]
        return [t.system(x + rng.normal(0.0, 0.005, x.shape), vel=vel, box=(63.0, 50.0, 50.0))]
    if case["path"] == REM:
        sizes, edges = water.replica_sizes(case["replicas"], seed=case["sizes"])
        return [water.water_box(int(m), float(L), seed=seed + k, jitter=0.2) for k, (m, L) in enumerate(zip(sizes, edges))]
    s = water.water_box(case["molecules"], round(_edge(case["molecules"]), 3), seed=seed, jitter=0.2)
    if case["path"] != RIGID:   # bonds and angles off their rest values
        s.pos = s.pos + rng.normal(0.0, 0.02, s.pos.shape)
    return [s]


def _lj_atoms(s, seed):
    """Per-atom sigma and epsilon of a parameter fit: the water's, 2 % off."""
    rng = np.random.default_rng([seed, 78])
    sigma = np.where(s.type == 0, water.SIGMA_O, 0.0) * (1.0 + 0.02 * rng.standard_normal(s.n))
    eps = np.where(s.type == 0, water.EPS_O, 0.0) * (1.0 + 0.02 * rng.standard_normal(s.n))
    return sigma, eps


def _alpha(rc, accuracy=1e-6):
    alpha = 1.0
    while math.erfc(alpha * rc) / rc >= accuracy:
        alpha *= 2.0
    lo, hi = 0.0, alpha
    for _ in range(100):
        alpha = 0.5 * (lo + hi)
        if math.erfc(alpha * rc) / rc >= accuracy:
            lo = alpha
        else:
            hi = alpha
    return alpha


def _field(case):
    """The force field of a case in plain values."""
    if case["path"] == PROTEIN:
        return dict(rc=10.0, on=0.1, alpha=0.312341327434087, pme_alpha=_alpha(10.0), grid=(60, 48, 48), order=4, cell=6.0,
                    coulomb="ewald")
    if case["path"] == REM:
        return dict(rc=8.0, on=7.0, alpha=0.0, grid=None, order=0, cell=4.0, coulomb="c2")
    rc = case["rc"]
    if case["field"] == "pme":
        return dict(rc=rc, on=rc - 1.0, alpha=_alpha(rc), pme_alpha=_alpha(rc), grid=(case["grid"],) * 3,
                    order=case["order"], cell=4.0, coulomb="ewald")
    return dict(rc=rc, on=rc - 1.0, alpha=0.0, grid=None, order=0, cell=4.0, coulomb="c1")


def _context(case, s, bonded=True):
    f = _field(case)
    ctx = gpu.Context(0, case["precision"])
    ctx.set_topology(s)
    ctx.set_boundary(s.box, s.origin, f["cell"])
    rc, on = f["rc"], f["on"]
    if f["coulomb"] == "ewald":
        hs = [ctx.force("LennardJones CoulombEwaldReal -algorithm NonbondedCutoff -switchingFunction C2 "
                        "-switchingFunction Cutoff", [on, rc, f["alpha"], rc, rc]),
              ctx.force("Coulomb -algorithm PMEwald -reciprocal -correction -interpolation BSpline",
                        [*f["grid"], rc, f["order"], 1e-6, -1.0])]
    else:
        hs = [ctx.force("LennardJones -algorithm NonbondedCutoff -switchingFunction C2", [on, rc, rc])]
        if f["coulomb"] == "c2":
            hs.append(ctx.force("Coulomb -algorithm NonbondedCutoff -switchingFunction C2", [on, rc, rc]))
        else:
            hs.append(ctx.force("Coulomb -algorithm NonbondedCutoff -switchingFunction C1", [rc, rc]))
    if bonded:
        hs += [ctx.force("Bond", []), ctx.force("Angle", [])]
        if case["path"] == PROTEIN:
            hs += [ctx.force("Dihedral", []), ctx.force("Improper", [])]
    return ctx, hs


def _dt(case):
    return 2.0 if case["path"] == RIGID else 1.0


def prepare(case, seed):
    boxes = _boxes(case, seed)
    path = case["path"]
    if path == REM:
        temps = water.replica_temperatures(case["replicas"])
        contexts = []
        for k, s in enumerate(boxes):
            ctx, hs = _context(case, s)
            ctx.md_setup(hs, "langevin", dt=1.0, temperature=float(temps[k]), gamma=5.0, seed=seed + k)
            ctx.md_set_state(s.pos, s.vel)
            contexts.append(ctx)
        return dict(case=case, batch=gpu.Batch(contexts), contexts=contexts, seed=seed, attempt=0)
    s = boxes[0]
    derivative = path in (HV, PARAM, LANCZOS)
    ctx, hs = _context(case, s, bonded=not derivative)
    st = dict(case=case, ctx=ctx, hs=hs, pos=s.pos, vel=s.vel)
    if path in (MD, RIGID, PROTEIN):
        ctx.md_setup(hs, "leapfrog", dt=_dt(case))
        ctx.md_set_state(s.pos, s.vel)
        if path == RIGID:
            ctx.md_set_constraints(1e-5, 30, 0.0, 0)
    if path in (HV, LANCZOS):
        st["v"] = np.random.default_rng([seed, 79]).standard_normal(s.pos.shape)
    if path == PARAM:
        ctx.set_lj_per_atom(*_lj_atoms(s, seed))
    return st


def run(state):
    case = state["case"]
    path = case["path"]
    if path == REM:
        batch = state["batch"]
        batch.run(case["steps"])
        _, deltas = batch.exchange(state["attempt"], state["seed"])
        state["attempt"] += 1
        ladder, _ = batch.ladder()
        got = [c.md_get_state() for c in state["contexts"]]
        x, v, e = (np.concatenate([g[k].reshape(-1) for g in got]) for k in range(3))
        return dict(x=x, v=v, energies=e, deltas=np.nan_to_num(deltas), ladder=ladder)
    ctx, hs = state["ctx"], state["hs"]
    if path == EVAL:
        f, e = ctx.evaluate(hs, state["pos"], virial=case["virial"])
        return dict(forces=f, energies=e)
    if path in (MD, RIGID, PROTEIN):
        ctx.md_set_state(state["pos"], state["vel"])
        ctx.md_run(case["steps"])
        x, v, e = ctx.md_get_state()
        return dict(x=x, v=v, energies=e)
    if path == HV:
        return dict(hv=ctx.hessian_vec(hs, state["pos"], state["v"]))
    if path == PARAM:
        dq, ds, de = ctx.param_gradients(hs, state["pos"])
        return dict(dq=dq, dsigma=ds, depsilon=de)
    vals, vecs, res, alpha, beta = ctx.lanczos(hs, state["pos"], state["v"], steps=case["steps"], nvec=min(20, case["steps"]),
                                               mass_weighted=True)
    return dict(values=vals, vectors=vecs, residuals=res, alpha=alpha, beta=beta)


# -------------------------------------------------------------------- work
def work(case):
    """Pairs within the cutoff at 69 flops each (61 with a plain Coulomb term;
    twice that for a second derivative), the grid's transforms, and each
    atom's state read and each result written once, for every force
    evaluation; the PME grid is written and read once by each of its passes."""
    f = _field(case)
    path = case["path"]
    if path == REM:
        n = 3 * int(water.replica_sizes(case["replicas"], seed=case["sizes"])[0].sum())
    else:
        n = 14281 if path == PROTEIN else 3 * case["molecules"]
    density = 14281 / (63.0 * 50.0 * 50.0) if path == PROTEIN else 3 * DENSITY
    pairs = n * density * (4.0 / 3.0) * math.pi * f["rc"] ** 3 / 2.0
    flops = pairs * (69.0 if f["coulomb"] == "ewald" else 61.0)
    word = 8 if case["precision"] == "double" else 4
    nbytes = n * (24 + 8 + 24.0)
    passes = 1
    if path in (HV, LANCZOS):
        flops *= 2.0
        passes = 2
    if f["grid"]:
        ng = f["grid"][0] * f["grid"][1] * f["grid"][2]
        ngc = f["grid"][0] * f["grid"][1] * (f["grid"][2] // 2 + 1)
        flops += passes * (2 * 2.5 * ng * math.log2(ng) + n * f["order"] ** 3 * 10.0)
        nbytes += passes * word * (4 * ng + 4 * ngc)
    evaluations = 1
    if path in (MD, RIGID, PROTEIN, REM):
        evaluations = case["steps"]
        nbytes += n * 72.0
        flops += n * 20.0
    if path == LANCZOS:
        evaluations = case["steps"]
        flops += 4.0 * 3 * n * case["steps"]
        nbytes += 8.0 * 3 * n * case["steps"] * 2
    return {"bytes": float(evaluations * nbytes), "flops": float(evaluations * flops)}


def tolerance(case):
    """About four times what a run is off 64 bits: FP32 pair and grid
    arithmetic (with exact integer sums of the forces) is 3e-7 to 2e-6 off in
    one evaluation, up to 9e-7 in velocities after tens of MD steps; FP64 1e-13
    to 1e-9 (an energy sum that nearly cancels).  A Lanczos run amplifies the
    product's rounding (3e-5 in mixed precision, 4e-11 in FP64), and so does
    the kick of a hot replica's closest contacts (6e-4 in velocities)."""
    mixed = case["precision"] == "mixed"
    path = case["path"]
    if path == REM:
        return {"rel": 2e-3, "max": 0.6, "differ": 0.0}
    if path in (MD, RIGID, PROTEIN):
        return {"rel": 4e-6 if mixed else 1e-11, "max": 4e-3 if mixed else 1e-8}
    if path == LANCZOS:
        return {"rel": 1.5e-4 if mixed else 2e-10, "max": 1e-2 if mixed else 1e-8}
    return {"rel": 1e-5 if mixed else 5e-9, "max": 1e-3 if mixed else 1e-7}


# ------------------------------------------------- the same in 64-bit torch
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


class _Exact:
    """Forces of one system, or of several boxes at once, in FP64."""

    def __init__(self, case, boxes, lj_atoms=None):
        d = self.d = _dev()
        self.f = _field(case)
        self.case = case

        def f64(a):
            return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=d)

        def i64(a):
            return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.int64, device=d)
        off = np.cumsum([0] + [s.n for s in boxes])
        self.off, self.n = off, int(off[-1])
        cat = lambda name: np.concatenate([getattr(s, name) for s in boxes])  # noqa: E731
        idx = lambda name: i64(np.concatenate([np.asarray(getattr(s, name)) + o for s, o in zip(boxes, off)]))  # noqa: E731
        self.q, self.type, self.mass = f64(cat("q")), i64(cat("type")), f64(cat("mass"))[:, None]
        self.L = f64(np.concatenate([np.tile(np.asarray(s.box, float), (s.n, 1)) for s in boxes]))
        s = boxes[0]
        self.A, self.B, self.A14, self.B14, self.csf = f64(s.ljA), f64(s.ljB), f64(s.ljA14), f64(s.ljB14), float(s.csf)
        self.lj_atoms = None if lj_atoms is None else tuple(f64(a) for a in lj_atoms)
        a, b, cls = idx("ex_a"), idx("ex_b"), i64(cat("ex_cls"))
        key = (torch.minimum(a, b) * self.n + torch.maximum(a, b)).cpu().numpy()
        # of a pair added more than once, the exclusion table holds the first
        # add (the correction's class), a look-up finds the last (the pair's)
        uniq, first = np.unique(key, return_index=True)
        last = len(key) - 1 - np.unique(key[::-1], return_index=True)[1]
        self.ex_key, self.ex_cls, self.ex_pair_cls = i64(uniq), cls[i64(first)], cls[i64(last)]
        self.ex_a, self.ex_b = self.ex_key // self.n, self.ex_key % self.n
        self.bonds = (idx("bond_a"), idx("bond_b"), f64(cat("bond_k")), f64(cat("bond_r0")))
        self.angles = (idx("angle_a"), idx("angle_b"), idx("angle_c"), f64(cat("angle_k")), f64(cat("angle_t0")),
                       f64(cat("angle_kub")), f64(cat("angle_rub")))
        self.torsions = []
        for name in ("dihedrals", "impropers"):
            t = getattr(s, name, None)
            if t is not None and len(t.atoms):
                row = np.repeat(np.arange(len(t.atoms)), np.diff(t.term_row))
                self.torsions.append((i64(t.atoms), i64(row), f64(t.k), f64(t.period), f64(t.phase)))
        self.bonded = case["path"] not in (HV, PARAM, LANCZOS)
        self.built = None
        self.skin = 1.0
        if self.f["grid"]:
            self._pme_setup(np.asarray(s.box, float))

    # pairs within the cutoff + skin, not fully excluded, i < j
    def _pairs(self, x):
        if self.built is not None:
            move = (x - self.built).square().sum(1).max().sqrt()
            if float(move) < 0.5 * self.skin:
                return self.pi, self.pj, self.pcls
        reach2 = (self.f["rc"] + self.skin) ** 2
        got_i, got_j = [], []

        def keep(i, j, L):
            dx = x[i] - x[j]
            dx = dx - L * torch.round(dx / L)
            ok = (dx.square().sum(-1) <= reach2) & (i < j)
            got_i.append(i[ok].int())
            got_j.append(j[ok].int())
        for k in range(len(self.off) - 1):
            lo, hi = int(self.off[k]), int(self.off[k + 1])
            L = self.L[lo]
            nc = (L / (self.f["rc"] + self.skin)).floor().long().tolist()
            atoms = torch.arange(lo, hi, device=self.d)
            if min(nc) < 3:
                step = max(1, 10_000_000 // (hi - lo))
                for c in range(lo, hi, step):
                    i = torch.arange(c, min(c + step, hi), device=self.d)[:, None].expand(-1, hi - lo)
                    keep(i, atoms[None].expand(i.shape[0], -1), L)
                continue
            n3 = torch.tensor(nc, device=self.d)
            u = x[lo:hi] / L
            c3 = torch.minimum(((u - u.floor()) * n3).long(), n3 - 1)
            cell = (c3[:, 0] * nc[1] + c3[:, 1]) * nc[2] + c3[:, 2]
            order = torch.argsort(cell, stable=True)
            count = torch.bincount(cell, minlength=nc[0] * nc[1] * nc[2])
            start = torch.cumsum(count, 0) - count
            m = int(count.max())
            table = torch.full((len(count), m), -1, dtype=torch.int64, device=self.d)
            cs = cell[order]
            table[cs, torch.arange(hi - lo, device=self.d) - start[cs]] = order + lo
            t4 = table.reshape(*nc, m)
            half = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]
            for o in half[half.index((0, 0, 0)):]:
                other = torch.roll(t4, shifts=(-o[0], -o[1], -o[2]), dims=(0, 1, 2)).reshape(-1, m)
                step = max(1, 20_000_000 // (m * m))
                for c in range(0, len(count), step):
                    i = table[c:c + step, :, None]
                    j = other[c:c + step, None, :]
                    dx = x[i.clamp(min=0)] - x[j.clamp(min=0)]
                    dx = dx - L * torch.round(dx / L)
                    ok = (dx.square().sum(-1) <= reach2) & (i >= 0) & (j >= 0)
                    if o == (0, 0, 0):
                        ok &= i < j
                    i, j = i.expand(ok.shape)[ok], j.expand(ok.shape)[ok]
                    got_i.append(torch.minimum(i, j).int())
                    got_j.append(torch.maximum(i, j).int())
        i, j = torch.cat(got_i), torch.cat(got_j)
        key = i.long() * self.n + j.long()
        at = torch.searchsorted(self.ex_key, key).clamp(max=len(self.ex_key) - 1)
        cls = torch.where(self.ex_key[at] == key, self.ex_pair_cls[at], torch.zeros_like(at)).to(torch.int8)
        ok = cls != 2
        self.pi, self.pj, self.pcls = i[ok], j[ok], cls[ok]
        self.built = x.clone()
        return self.pi, self.pj, self.pcls

    def _swf(self, kind, r2):
        f = self.f
        c2, on2 = f["rc"] ** 2, f["on"] ** 2
        if kind == "c2":
            d = c2 - r2
            m = d * (c2 - 3.0 * on2 + 2.0 * r2)
            w = (c2 - on2) ** 3
            inside = r2 < on2
            return (torch.where(inside, torch.ones_like(r2), d * m / w),
                    torch.where(inside, torch.zeros_like(r2), 4.0 / w * (d * d - m)))
        r, c = r2.sqrt(), f["rc"]
        return 1.0 - r * (1.5 / c - r2 * 0.5 / c ** 3), -1.5 / c / r + r * 1.5 / c ** 3

    def _pair(self, r2, qq, A, B):
        """Energies (Lennard-Jones, Coulomb) and force / r of pairs at r2 <= rc^2."""
        rr2 = 1.0 / r2
        r6 = rr2 * rr2 * rr2
        e_lj = A * r6 * r6 - B * r6
        f_lj = (12.0 * A * r6 * r6 - 6.0 * B * r6) * rr2
        s, ds = self._swf("c2", r2)
        f_lj, e_lj = f_lj * s - e_lj * ds, e_lj * s
        if self.f["coulomb"] == "ewald":
            al = self.f["alpha"]
            r = r2.sqrt()
            ar = al * r
            t = 1.0 / (1.0 + 0.3275911 * ar)
            p = t * (0.254829592 + t * (-0.284496736 + t * (1.421413741 + t * (-1.453152027 + t * 1.061405429))))
            g = qq * torch.exp(-ar * ar)
            e_c = p * g / r
            f_c = (e_c + 2.0 * al / math.sqrt(math.pi) * g) * rr2
        else:
            e = qq * rr2.sqrt()
            s, ds = self._swf(self.f["coulomb"], r2)
            f_c, e_c = e * rr2 * s - e * ds, e * s
        return e_lj, e_c, f_lj + f_c

    def _chunks(self, x, size=4_000_000):
        """(i, j, displacement x_j - x_i, charge product, A, B, class) of the pairs within the cutoff."""
        pi, pj, pc = self._pairs(x)
        for c in range(0, len(pi), size):
            i, j, cls = pi[c:c + size].long(), pj[c:c + size].long(), pc[c:c + size]
            L = self.L[i]
            d = x[j] - x[i]
            d = d - L * torch.round(d / L)
            ok = d.square().sum(1) <= self.f["rc"] ** 2
            i, j, d, cls = i[ok], j[ok], d[ok], cls[ok]
            mod = cls == 1
            ti, tj = self.type[i], self.type[j]
            A = torch.where(mod, self.A14[ti, tj], self.A[ti, tj])
            B = torch.where(mod, self.B14[ti, tj], self.B[ti, tj])
            qq = self.q[i] * self.q[j] * torch.where(mod, self.csf, 1.0).to(torch.float64)
            yield i, j, d, qq, A, B

    # particle-mesh Ewald
    def _pme_setup(self, box):
        f = self.f
        n = f["grid"]
        al = f["pme_alpha"]
        m = [torch.fft.fftfreq(n[0], 1.0 / n[0]), torch.fft.fftfreq(n[1], 1.0 / n[1]), torch.arange(n[2] // 2 + 1)]
        m = [(v.to(torch.float64) / L).to(self.d) for v, L in zip(m, box)]
        w0 = self._spline(torch.zeros(1, dtype=torch.float64, device=self.d))[0]
        mod = []
        for a in range(3):
            k = torch.arange(n[a], dtype=torch.float64, device=self.d)[:, None]
            ph = 2.0 * math.pi * k * torch.arange(f["order"], dtype=torch.float64, device=self.d) / n[a]
            b = 1.0 / ((w0 * torch.cos(ph)).sum(1) ** 2 + (w0 * torch.sin(ph)).sum(1) ** 2)
            mod.append(b[:len(m[a])])
        m2 = m[0][:, None, None] ** 2 + m[1][None, :, None] ** 2 + m[2][None, None] ** 2
        m2[0, 0, 0] = 1.0
        self.fac = (math.pi / al) ** 2
        V = float(np.prod(box))
        th = torch.exp(-self.fac * m2) / (math.pi * V) / m2 * mod[0][:, None, None] * mod[1][None, :, None] * mod[2][None, None]
        th[0, 0, 0] = 0.0
        self.m, self.m2 = m, m2
        # both halves of the spectrum: kz of 0 and, for an even size, n/2 stand once
        both = torch.full((n[2] // 2 + 1,), 2.0, dtype=torch.float64, device=self.d)
        both[0] = 1.0
        if n[2] % 2 == 0:
            both[-1] = 1.0
        self.theta = th * both
        self.box = box
        self.n_over_L = torch.tensor([g / L for g, L in zip(n, box)], dtype=torch.float64, device=self.d)

    def _spline(self, w):
        """B-spline weights (..., order) at fractional offsets w, by the recursion in the order."""
        th = [1.0 - w, w]
        for k in range(3, self.f["order"] + 1):
            new = []
            for j in range(k):
                # M_k at u = w + (k - 1 - j): the weights stand in falling order of u
                u = w + (k - 1 - j)
                left = th[j - 1] if j > 0 else 0.0     # M_{k-1}(u)
                right = th[j] if j < k - 1 else 0.0    # M_{k-1}(u - 1)
                new.append((u * left + (k - u) * right) / (k - 1))
            th = new
        return torch.stack(th, -1)

    def _recip(self, x, q, parts=False):
        """The reciprocal energy (with the virial where asked)."""
        n = self.f["grid"]
        p = self.f["order"]
        u = x * self.n_over_L
        i0 = u.detach().floor()
        w = u - i0
        th = [self._spline(w[:, a]) for a in range(3)]
        at = [torch.remainder(i0[:, a].long()[:, None] - (p - 1) // 2 + torch.arange(p, device=self.d), n[a]) for a in range(3)]
        Q = torch.zeros(n[0] * n[1] * n[2], dtype=torch.float64, device=self.d)
        for a in range(p):
            for b in range(p):
                row = (at[0][:, a] * n[1] + at[1][:, b])[:, None] * n[2] + at[2]
                val = (q * th[0][:, a] * th[1][:, b])[:, None] * th[2]
                Q = Q.index_add(0, row.reshape(-1), val.reshape(-1))
        S = torch.fft.rfftn(Q.reshape(n))
        e = self.theta * (S.real.square() + S.imag.square())
        if not parts:
            return 0.5 * e.sum()
        vir = torch.zeros(3, 3, dtype=torch.float64, device=self.d)
        vv = 2.0 * (1.0 / self.m2 + self.fac)
        mm = [self.m[0][:, None, None], self.m[1][None, :, None], self.m[2][None, None]]
        # the products of mixed sign cancel between the halves that stand twice and add up once for the planes that stand once
        for a in range(3):
            for b in range(3):
                vir[a, b] = 0.5 * (e * ((1.0 if a == b else 0.0) - vv * mm[a] * mm[b])).sum()
        return 0.5 * e.sum(), vir

    def _corr(self, x, q):
        """Energy of the excluded pairs' correction, and their force / r and displacements."""
        qq = q[self.ex_a] * q[self.ex_b] * torch.where(self.ex_cls == 1, 1.0 - self.csf, 1.0).to(torch.float64)
        d = x[self.ex_b] - x[self.ex_a]
        d = d - (self.L[self.ex_a] * torch.round(d / self.L[self.ex_a])).detach()
        r = d.square().sum(1).sqrt()
        return -(qq * torch.erf(self.f["pme_alpha"] * r) / r).sum(), d

    def _self(self, q):
        al, V = self.f["pme_alpha"], float(np.prod(self.box))
        e = -(q * q).sum() * al / math.sqrt(math.pi)
        net = q.sum()
        charged = -math.pi / (2.0 * V * al * al) * net * net if abs(float(net.detach()) * 0.00268283) > 1.0e-5 else 0.0 * net
        return e, charged

    def _min(self, x, a, b):
        d = x[a] - x[b]
        return d - self.L[a] * torch.round(d / self.L[a])

    def forces(self, x, virial=False):
        """Forces (n, 3) and the energy record of 16, of every box together."""
        F = torch.zeros_like(x)
        boxes = len(self.off) - 1
        E = torch.zeros(boxes, 16, dtype=torch.float64, device=self.d)
        W = torch.zeros(3, 3, dtype=torch.float64, device=self.d)
        atom = torch.zeros(4, self.n, dtype=torch.float64, device=self.d)   # Coulomb, LJ, bond, angle energies by an atom
        for i, j, d, qq, A, B in self._chunks(x):
            el, ec, f = self._pair(d.square().sum(1), qq, A, B)
            fd = d * f[:, None]
            F.index_add_(0, j, fd)
            F.index_add_(0, i, -fd)
            atom[0].index_add_(0, i, ec)
            atom[1].index_add_(0, i, el)
            if virial:
                W += fd.T @ d
        if self.f["grid"]:
            xg = x.detach().clone().requires_grad_(True)
            with torch.enable_grad():
                e, vir = self._recip(xg, self.q, parts=True)
                ec, d = self._corr(xg, self.q)
                gr, = torch.autograd.grad(e, xg, retain_graph=True)
                gc, gd = torch.autograd.grad(ec, (xg, d))
            F -= gr + gc
            es, ech = self._self(self.q)
            E[0, 0] += e.detach() + ec.detach() + es + ech
            W += vir.detach() - gd.T @ d.detach() + ech * torch.eye(3, dtype=torch.float64, device=self.d)
        if self.bonded:
            a, b, k, r0 = self.bonds
            d = self._min(x, a, b)
            r = d.square().sum(1).sqrt()
            f = -(2.0 * k * (r - r0) / r)[:, None] * d
            F.index_add_(0, a, f)
            F.index_add_(0, b, -f)
            atom[2].index_add_(0, a, k * (r - r0) ** 2)
            W += f.T @ d
            self._angles(x, F, atom[3], W)
            for t, kind in zip(self.torsions, (4, 5)):
                self._torsions(x, t, kind, F, E, W)
        for k in range(boxes):
            E[k, :4] += atom[:, int(self.off[k]):int(self.off[k + 1])].sum(1)
        if virial:
            E[0, 7:16] = W.reshape(-1)
        return F, E

    def _angles(self, x, F, atom, W):
        a, b, c, k, t0, kub, rub = self.angles
        with torch.enable_grad():
            d1 = self._min(x, a, b).detach().requires_grad_(True)
            d3 = self._min(x, c, b).detach().requires_grad_(True)
            theta = torch.atan2(torch.linalg.cross(d1, d3).norm(dim=1), (d1 * d3).sum(1))
            e = k * (theta - t0) ** 2
            if bool((kub != 0).any()):
                e = e + kub * ((d1 - d3).square().sum(1).sqrt() - rub) ** 2
            g1, g3 = torch.autograd.grad(e.sum(), (d1, d3))
        F.index_add_(0, a, -g1)
        F.index_add_(0, c, -g3)
        F.index_add_(0, b, g1 + g3)
        atom.index_add_(0, a, e.detach())
        W -= g1.T @ d1.detach() + g3.T @ d3.detach()

    def _torsions(self, x, t, kind, F, E, W):
        at, row, k, period, phase = t
        with torch.enable_grad():
            d = [self._min(x, at[:, u], at[:, u + 1]).detach().requires_grad_(True) for u in range(3)]
            na, nb = torch.linalg.cross(d[0], d[1]), torch.linalg.cross(d[1], d[2])
            nc = torch.linalg.cross(d[1], na)
            unit = lambda v: v / v.norm(dim=1, keepdim=True)  # noqa: E731
            phi = -torch.atan2((unit(nc) * unit(nb)).sum(1), (unit(na) * unit(nb)).sum(1))[row]
            diff = phi - phase
            diff = diff - 2.0 * math.pi * torch.round(diff.detach() / (2.0 * math.pi))
            e = torch.where(period > 0, k * (1.0 + torch.cos(period * phi + phase)), k * diff * diff)
            g = torch.autograd.grad(e.sum(), d)
        for u in range(3):
            F.index_add_(0, at[:, u], -g[u])
            F.index_add_(0, at[:, u + 1], g[u])
            W -= g[u].T @ d[u].detach()
        E[0, kind] += e.detach().sum()

    def hessian_vec(self, x, v):
        out = torch.zeros_like(x)
        for i, j, d, qq, A, B in self._chunks(x):
            fn = lambda d: d * self._pair(d.square().sum(1), qq, A, B)[2][:, None]  # noqa: E731
            _, t = torch.func.jvp(fn, (d,), (v[j] - v[i],))
            out.index_add_(0, j, -t)
            out.index_add_(0, i, t)
        if self.f["grid"]:
            xg = x.detach().clone().requires_grad_(True)
            with torch.enable_grad():
                e = self._recip(xg, self.q) + self._corr(xg, self.q)[0]
                g, = torch.autograd.grad(e, xg, create_graph=True)
                h, = torch.autograd.grad((g * v).sum(), xg)
            out += h
        return out

    def param_gradients(self, x):
        q = self.q.clone().requires_grad_(True)
        sigma, eps = (a.clone().requires_grad_(True) for a in self.lj_atoms)
        total = [torch.zeros_like(q) for _ in range(3)]
        for i, j, d, _, _, _ in self._chunks(x):
            with torch.enable_grad():
                r2 = d.square().sum(1)
                # atoms without Lennard-Jones have no such pairs (and no gradient there)
                on = (eps.detach()[i] > 0) & (eps.detach()[j] > 0)
                R = (sigma[i] + sigma[j]) * 2.0 ** (-5.0 / 6.0)
                w = torch.where(on, eps[i] * eps[j], torch.ones_like(R)).sqrt() * on
                e_lj, e_c, _ = self._pair(r2, q[i] * q[j], R ** 12 * w, 2.0 * R ** 6 * w)
                got = torch.autograd.grad(e_lj.sum() + e_c.sum(), (q, sigma, eps))
            total = [t + g for t, g in zip(total, got)]
        if self.f["grid"]:
            with torch.enable_grad():
                es, ech = self._self(q)
                e = self._recip(x, q) + self._corr(x, q)[0] + es + ech
                total[0] = total[0] + torch.autograd.grad(e, q)[0]
        return total


def _shake(m, x, v, last, eps=1e-5, most=30, dt=2.0):
    """SHAKE of the waters (O, H, H): sweeps over O-H, O-H, H-H until the mean error is within eps."""
    hh = math.sqrt(2.0 * water.R_OH ** 2 * (1.0 - math.cos(math.radians(water.THETA_HOH))))
    cons = [(0, 1, water.R_OH), (0, 2, water.R_OH), (1, 2, hh)]
    x, v, last = (t.reshape(-1, 3, 3).clone() for t in (x, v, last))
    m = m.reshape(-1, 3)

    def error():
        return float(sum(((x[:, b] - x[:, a]).square().sum(1) - r * r).abs().sum() / (2.0 * r * r)
                         for a, b, r in cons) / (3 * len(x)))
    sweeps = 0
    while error() > eps:
        for a, b, r in cons:
            p, o = x[:, a] - x[:, b], last[:, a] - last[:, b]
            wa, wb = 1.0 / m[:, a], 1.0 / m[:, b]
            g = (r * r - p.square().sum(1)) / (2.0 * (wa + wb) * (o * p).sum(1))
            dp = o * g[:, None]
            x[:, a] += dp * wa[:, None]
            x[:, b] -= dp * wb[:, None]
            v[:, a] += dp * wa[:, None] / (dt * TIME)
            v[:, b] -= dp * wb[:, None] / (dt * TIME)
        sweeps += 1
        if sweeps > most:
            break
    return x.reshape(-1, 3), v.reshape(-1, 3)


_M64 = (1 << 64) - 1


def _mix64(z):
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


def _noise(seed, counter, n3):
    """The Gaussian deviates of a Langevin half kick (SplitMix64 of seed, counter and index, Box-Muller)."""
    idx = np.arange(n3, dtype=np.uint64)
    with np.errstate(over="ignore"):
        h1 = _mix64(np.uint64(seed) ^ _mix64(np.uint64((counter * 0x100000001B3) & _M64) + idx * np.uint64(2)))
    h2 = _mix64(h1 ^ np.uint64(0x5851F42D4C957F2D))
    u1 = ((h1 >> np.uint64(11)) + np.uint64(1)).astype(np.float64) * (1.0 / 9007199254740993.0)
    u2 = (h2 >> np.uint64(11)).astype(np.float64) * (1.0 / 9007199254740992.0)
    return np.sqrt(-2.0 * np.log(u1)) * np.cos(6.283185307179586 * u2)


def _exact_replicas(case, boxes, seed):
    """One exchange interval: Langevin leapfrog of every box, then the test of neighbours on the ladder."""
    ex = _Exact(case, boxes)
    R = len(boxes)
    temps = water.replica_temperatures(R)
    d = ex.d
    x = torch.as_tensor(np.concatenate([s.pos for s in boxes]), device=d)
    v = torch.as_tensor(np.concatenate([s.vel for s in boxes]), device=d)
    T = torch.as_tensor(np.repeat(temps, np.diff(ex.off)), device=d)[:, None]
    h = TIME
    g = 5.0 / (1000.0 * TIME)
    fdt, vdt = (1.0 - math.exp(-0.5 * g * h)) / g, math.exp(-0.5 * g * h)
    ndt = math.sqrt((1.0 - math.exp(-g * h)) / (2.0 * g))
    scale = torch.sqrt(2.0 * KB * T * g / ex.mass) * ndt
    counter = 0

    def kick():
        nonlocal counter, v
        xi = np.concatenate([_noise(seed + k, counter, 3 * s.n).reshape(-1, 3) for k, s in enumerate(boxes)])
        counter += 1
        v = v * vdt + F * fdt / ex.mass + torch.as_tensor(xi, device=d) * scale
    F, E = ex.forces(x)
    for _ in range(case["steps"]):
        kick()
        x = x + v * h
        F, E = ex.forces(x)
        kick()
    pot = E[:, :7].sum(1).cpu().numpy()
    ladder, deltas = np.arange(R, dtype=np.int32), np.zeros(R)
    for k in range(0, R - 1, 2):
        delta = (1.0 / KB / temps[k] - 1.0 / KB / temps[k + 1]) * (pot[k + 1] - pot[k])
        h = _mix64(np.uint64(seed) ^ _mix64(np.uint64(2 * k + 1)))   # attempt 0
        u = float(h >> np.uint64(11)) / 9007199254740992.0
        deltas[k] = delta
        if u <= (1.0 if delta <= 0 else math.exp(-delta)):
            ladder[k], ladder[k + 1] = k + 1, k
            for r, t in ((k, temps[k + 1] / temps[k]), (k + 1, temps[k] / temps[k + 1])):
                v[ex.off[r]:ex.off[r + 1]] *= math.sqrt(t)
    return dict(x=x.reshape(-1), v=v.reshape(-1), energies=E.reshape(-1), deltas=deltas, ladder=ladder)


@torch.no_grad()
def exact(case, seed):
    boxes = _boxes(case, seed)
    path = case["path"]
    if path == REM:
        return _exact_replicas(case, boxes, seed)
    s = boxes[0]
    ex = _Exact(case, boxes, _lj_atoms(s, seed) if path == PARAM else None)
    x = torch.as_tensor(s.pos, device=ex.d)
    if path == EVAL:
        F, E = ex.forces(x, virial=case["virial"])
        return dict(forces=F, energies=E[0])
    if path == PARAM:
        dq, ds, de = ex.param_gradients(x)
        return dict(dq=dq, dsigma=ds, depsilon=de)
    if path in (HV, LANCZOS):
        v = torch.as_tensor(np.random.default_rng([seed, 79]).standard_normal(s.pos.shape), device=ex.d)
        if path == HV:
            return dict(hv=ex.hessian_vec(x, v))
        steps = case["steps"]
        w = 1.0 / ex.mass.sqrt()
        V = torch.zeros(steps + 1, x.numel(), dtype=torch.float64, device=ex.d)
        V[0] = v.reshape(-1) / v.norm()
        alpha, beta = np.zeros(steps), np.zeros(steps)
        for k in range(steps):
            u = (w * ex.hessian_vec(x, w * V[k].reshape(-1, 3))).reshape(-1)
            for _ in range(2):
                c = V[:k + 1] @ u
                u = u - c @ V[:k + 1]
                alpha[k] += float(c[k])
            beta[k] = float(u.norm())
            V[k + 1] = u / beta[k]
        vals, vecs = np.linalg.eigh(np.diag(alpha) + np.diag(beta[:-1], 1) + np.diag(beta[:-1], -1))
        # the sign of a vector is free
        return dict(values=vals, vectors=None, residuals=np.abs(beta[-1] * vecs[-1]), alpha=alpha, beta=beta)
    # leapfrog: half kick and drift, forces, kicks and drifts, half kick
    v = torch.as_tensor(s.vel, device=ex.d)
    h = _dt(case) * TIME
    last = x
    F, E = ex.forces(x)
    for k in range(case["steps"]):
        v = v + F * (h * (0.5 if k == 0 else 1.0)) / ex.mass
        x = x + v * h
        if path == RIGID:
            x, v = _shake(ex.mass[:, 0], x, v, last)
            last = x
        F, E = ex.forces(x)
    v = v + F * (0.5 * h) / ex.mass
    return dict(x=x, v=v, energies=E[0])
