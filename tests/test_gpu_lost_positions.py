"""Positions that are lost between the neighbour lists and the passes that walk
them: infinite by a density fix with an infinite velocity (particles.h:303-305),
NaN by a NaN multiplier or a position star the caller wrote.  The distance to
the far row that pads the lists is a NaN for most of them, which the test for a
neighbour within h keeps (particles.h:307), so the walk of such a particle has
to end at its count: no term of the padding enters a sum, and its compact row
stays within its bounds.

The library is compared with the passes written out in numpy, entry by entry in
list order, pairs farther than h left out.  (Not with the oracle where a NaN
spreads: it adds a factor of zero for those pairs, which is a NaN where the
other factor is one.)  On finite scenes they agree with the oracle: the CPU
test.  All bit for bit, NaN where the other has NaN.  List caps on and off the
multiples of eight and sixteen entries."""
import os

import numpy as np
import pytest

import oracle_lib as O

THREADS = max(1, min(16, os.cpu_count() or 1))
F = np.float32

# (lanes a particle in the pressure solve, the passes after it, the passes
# one by one: 16, 16, 4 up to 4,099; 4, 16, 4 at 20,000; 4, 4, 4 at 40,000;
# 1, 4, 1 at 160,000; 1, 1, 1 at 530,000)
SIZES = [(2, 7), (300, 1), (1000, 8), (1000, 40), (4099, 7), (4099, 60), (4099, 128), (20000, 100), (20000, 1),
         (40000, 7), (40000, 60), (160000, 40), (530000, 7)]


class Model:
    """The passes in float32, one list entry of all particles at a time."""

    def __init__(self, p, x, v):
        self.p, self.x, self.v, self.xs = p, x.copy(), v.copy(), x.copy()
        self.rho, self.lam, self.scr = (np.zeros(s, F) for s in (len(x), len(x), x.shape))
        self.h, self.dt, self.rho0, self.mass = F(p.smoothing_radius), F(p.time_step), F(p.rest_density), F(p.rest_mass)
        self.poly6_norm = F(315.0 / (64.0 * np.pi * float(self.h) ** 9.0))
        self.spiky_norm = F(-45.0 / (np.pi * float(self.h) ** 6.0))
        self.eps = np.finfo(F).eps

    def lists(self, nbr, cnt):
        self.nbr, self.cnt = nbr.astype(np.int64), cnt

    @staticmethod
    def magsq(a):
        return ((a[:, 0] * a[:, 0] + a[:, 1] * a[:, 1]) + a[:, 2] * a[:, 2]).astype(F)

    def poly6(self, r):
        w = self.h * self.h - r * r
        return self.poly6_norm * w * w * w

    def spiky(self, d, r):
        return ((self.spiky_norm * (self.h - r) * (self.h - r))[:, None] * d) / (r + self.eps)[:, None]

    def pairs(self, pos):
        """(p, q, d, r) of every entry within h, entry by entry"""
        for k in range(int(self.cnt.max(initial=0))):
            i = np.nonzero(k < self.cnt)[0]
            q = self.nbr[i, k]
            d = pos[i] - pos[q]
            r = np.sqrt(self.magsq(d))
            m = ~(r > self.h)
            yield i[m], q[m], d[m], r[m]

    def boundary(self, a):
        p = self.p
        c = np.array(p.mover_center[:], F)
        d2 = self.magsq(a - c)
        m = d2 < F(0.2) * F(0.2)
        r = np.sqrt(d2[m])
        a[m] += ((F(0.2) - r)[:, None] * (a[m] - c)) / r[:, None]
        for i in range(3):
            lo, hi = F(p.boundary_min[i]), F(p.boundary_max[i])
            low, high = a[:, i] < lo, a[:, i] > hi
            a[low, i], a[high, i] = lo, hi

    def forces_predict(self):
        self.v[:, 1] += F(self.p.gravity) * self.dt
        self.xs = self.x + self.v * self.dt
        self.boundary(self.xs)

    def density(self):
        rho = np.full(len(self.x), self.mass * (self.poly6_norm * (self.h * self.h) * (self.h * self.h) * (self.h * self.h)), F)
        at, moved = self.xs, self.xs.copy()
        self.hacks = 0
        for k in range(int(self.cnt.max(initial=0))):
            i = np.nonzero(k < self.cnt)[0]
            q = self.nbr[i, k]
            near = np.sqrt(self.magsq(moved[i] - at[q])).astype(np.float64) < 0.00000001
            j = i[near]
            moved[j] -= (self.v[j] * self.dt) / F(50.0)
            self.hacks += len(j)
            r = np.sqrt(self.magsq(moved[i] - at[q]))
            m = ~(r > self.h)
            rho[i[m]] += self.mass * self.poly6(r[m])
        self.rho, self.xs = rho, moved

    def multipliers(self):
        sg, sc = np.zeros_like(self.x), np.zeros(len(self.x), F)
        for i, q, d, r in self.pairs(self.xs):
            g = (F(-1.0) / self.rho0) * self.spiky(d, r)
            sg[i] -= g
            sc[i] += self.magsq(g)
        sc += self.magsq(sg)
        c = self.rho / self.rho0 - F(1.0)
        self.lam = -np.where(c < 0.0, F(0.0), c) / (sc + F(self.p.lambda_epsilon))

    def dps(self):
        dp = np.zeros_like(self.x)
        for i, q, d, r in self.pairs(self.xs):
            dp[i] += (self.lam[i] + self.lam[q])[:, None] * self.spiky(d, r)
        self.scr = (F(1.0) / self.rho0) * dp

    def stars(self):
        self.xs = self.xs + self.scr
        self.boundary(self.xs)

    def velocities(self):
        v = (self.xs - self.x) / self.dt
        v[self.magsq(v).astype(np.float64) < 0.000001 * float(F(self.p.max_speed))] = 0
        self.v = v

    def viscosity(self):
        dv = np.zeros_like(self.x)
        for i, q, d, r in self.pairs(self.xs):
            dv[i] += ((self.v[q] - self.v[i]) * self.poly6(r)[:, None]) / self.rho[q][:, None]
        self.v = self.v + F(self.p.visc_c) * dv

    @staticmethod
    def cross(a, b):
        return np.stack([a[:, 1] * b[:, 2] - a[:, 2] * b[:, 1], a[:, 2] * b[:, 0] - a[:, 0] * b[:, 2],
                         a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]], 1)

    def vorticity(self):
        w = np.zeros_like(self.x)
        for i, q, d, r in self.pairs(self.xs):
            w[i] += self.cross(self.v[q] - self.v[i], self.spiky(d, r))
        self.scr = w

    def confinement(self):
        eta, wm = np.zeros_like(self.x), np.sqrt(self.magsq(self.scr))
        for i, q, d, r in self.pairs(self.xs):
            eta[i] += wm[q][:, None] * self.spiky(d, r)
        N = eta / (np.sqrt(self.magsq(eta)) + self.eps)[:, None]
        self.v = self.v + (self.cross(N, self.scr) * F(self.p.vorticity_coef)) * self.dt

    def tail(self):
        for f in (self.velocities, self.viscosity, self.vorticity, self.confinement, self.viscosity):
            f()
        self.x = self.xs.copy()

    def state(self):
        return {"x": self.x, "xs": self.xs, "v": self.v, "rho": self.rho, "lam": self.lam, "scratch": self.scr}


@pytest.fixture(autouse=True)
def _quiet():
    with np.errstate(all="ignore"):
        yield


def _same(a, b):
    b = np.asarray(b).astype(F)
    return (a == b) | (np.isnan(a) & np.isnan(b))


def _compare(g, s, what, scratch=False):
    got = [("position stars", g.position_stars(), s["xs"]), ("velocities", g.velocities(), s["v"]),
           ("densities", g.densities(), s["rho"]), ("lambdas", g.lambdas(), s["lam"]),
           ("positions", g.positions(), s["x"])]
    if scratch:
        got.append(("scratch", g.scratch(), s["scratch"]))
    for name, a, b in got:
        bad = ~_same(a, b)
        assert not bad.any(), f"{what}: {name}: {int(bad.sum())} differ, first {np.argwhere(bad)[:3].tolist()}"


def _points(n, cap):
    """Random points, 8 to a cube of edge h."""
    side = max(0.2, (n / 8000.0) ** (1 / 3))
    return np.random.default_rng(n + cap).uniform(0.02, side, size=(n, 3)).astype(F), side + 0.1


def _thrown(n, cap):
    """Points on the low and high walls of x, y and z, each with another thrown
    onto it with an infinite velocity: the two coincide, and the density fix
    takes the thrown one through the box to the other infinity."""
    pos, side = _points(n, cap)
    vel = np.zeros_like(pos)
    pairs = max(1, min(n // 16, 40))
    for i in range(pairs):
        a, high, j = i % 3, (i // 3) % 2, n - pairs + i
        pos[j] = pos[i]
        pos[i, a] = F(side) if high else 0.0
        vel[j, a] = np.inf if high else -np.inf
    return pos, vel, side


def _params(pbf, scenes, n, cap, side, options=0, iters=4):
    p = scenes.pbf_params((side,) * 3, n, cap=cap, iters=iters, gravity=0.0)
    p.options |= options
    return p


@pytest.mark.parametrize("n,cap", [(1, 4), (700, 7), (3000, 60)])
def test_the_written_passes_are_the_oracles(pbf, scenes, n, cap):
    pos, side = _points(n, cap)
    pos[-(n // 8) - 1:] = pos[:n // 8 + 1]
    vel = np.random.default_rng(n).normal(0, 0.5, pos.shape).astype(F)
    p = scenes.pbf_params((side,) * 3, n, cap=cap)
    m = Model(p, pos, vel)
    o = O.Oracle(O.params_from_pbf(p), mode=O.JACOBI, threads=THREADS)
    o.set_state(pos, pos, vel)
    m.forces_predict()
    for i in (O.FORCES, O.PREDICT, O.FIND):
        o.pass_(i)
    m.lists(o.neighbors()["lists"], o.neighbors()["counts"])
    todo = [(m.density, O.DENSITY), (m.multipliers, O.LAMBDA), (m.dps, O.DP), (m.stars, O.UPDATE_XS)] * 2 + [
        (m.velocities, O.UPDATE_V), (m.viscosity, O.VISC), (m.vorticity, O.VORT), (m.confinement, O.APPLY_VORT),
        (m.viscosity, O.VISC)]
    hacks = 0
    for f, i in todo:
        f()
        hacks += m.hacks if i == O.DENSITY else 0
        o.pass_(i)
        s = o.state()
        for k in ("xs", "v", "rho", "lam", "scratch"):
            assert _same(m.state()[k], s[k]).all(), (f.__name__, k)
    assert hacks == o.counters()["hacks"]


@pytest.mark.gpu
@pytest.mark.parametrize("options,n,cap", [(o, n, cap) for o, most in (("none", 10**6), ("full_lists", 200000), ("persistent", 20000))
                                           for n, cap in SIZES if n <= most])
def test_density_fix_to_infinity(pbf, scenes, options, n, cap):
    """The thrown particles are lost between the density pass and the pressure
    update, which clamps them onto the box (unless they met another one)."""
    bits = {"none": 0, "full_lists": pbf.PBF_OPT_FULL_LISTS, "persistent": pbf.PBF_OPT_PERSISTENT}[options]
    pos, vel, side = _thrown(n, cap)
    p = _params(pbf, scenes, n, cap, side, bits)
    g = pbf.Particles(p)
    g.add(pos, pos, vel)
    m = Model(p, pos, vel)
    for step in range(2):
        g.step(1)
        m.forces_predict()
        m.lists(*g.neighbor_lists())
        hacks = 0
        for _ in range(p.solve_step_count):
            m.density()
            hacks += m.hacks
            m.multipliers()
            m.dps()
            m.stars()
        m.tail()
        _compare(g, m.state(), f"step {step + 1}")
        assert hacks == g.stats()["density_hacks"]
        assert hacks > 0 or cap < 40 or step


@pytest.mark.gpu
@pytest.mark.parametrize("n,cap", SIZES)
def test_infinite_to_the_end_of_the_step(pbf, scenes, n, cap):
    """A solve whose first density pass meets the tolerance makes no pressure
    update: what the density fix lost goes through the XSPH and vorticity passes."""
    pos, vel, side = _thrown(n, cap)
    p = _params(pbf, scenes, n, cap, side)
    g = pbf.Particles(p)
    g.add(pos, pos, vel)
    m = Model(p, pos, vel)
    g.solve(1e30, 3)
    m.forces_predict()
    m.lists(*g.neighbor_lists())
    m.density()
    m.multipliers()
    assert g.solve_info()["iterations"] == 1 and g.stats()["density_hacks"] == m.hacks
    assert np.isinf(m.xs).any() or cap < 40
    m.tail()
    _compare(g, m.state(), "solve")


@pytest.mark.gpu
@pytest.mark.parametrize("n,cap", SIZES)
def test_nan_multiplier_in_a_solve(pbf, scenes, n, cap):
    """Multipliers given as a warm start, one NaN and one infinite: the
    particles around them are lost from then on to the step's end."""
    pos, side = _points(n, cap)
    vel = np.zeros_like(pos)
    p = _params(pbf, scenes, n, cap, side, pbf.PBF_OPT_FULL_LISTS)
    g = pbf.Particles(p)
    g.add(pos, pos, vel)
    m = Model(p, pos, vel)
    warm = np.full(n, -1e-5, F)
    warm[n // 2] = np.nan
    warm[n // 3] = np.inf
    g.set_warm_lambdas(warm)
    g.solve(0.0, 3, pbf.PBF_WARM_GIVEN)
    m.forces_predict()
    m.lists(*g.neighbor_lists())
    m.density()
    before = m.xs.copy()
    m.lam = warm
    m.dps()
    m.stars()
    info = g.solve_info()
    assert np.isnan(m.xs).any() or cap < 40
    for it in range(info["iterations"]):
        m.density()
        m.multipliers()
        if it == 0 and not info["warm_start_kept"]:
            m.xs = before
        elif info["max_error_history"][it] > 0:
            m.dps()
            m.stars()
    m.tail()
    _compare(g, m.state(), "solve")


@pytest.mark.gpu
@pytest.mark.parametrize("n,cap", SIZES)
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_lost_in_the_passes(pbf, scenes, n, cap, value):
    """The passes one by one, position stars written over after the lists."""
    pos, side = _points(n, cap)
    vel = np.random.default_rng(n).normal(0, 0.1, pos.shape).astype(F)
    p = _params(pbf, scenes, n, cap, side)
    g = pbf.Particles(p)
    g.add(pos, pos, vel)
    m = Model(p, pos, vel)
    g.apply_external_forces()
    g.predict_positions()
    g.find_neighbors()
    m.forces_predict()
    m.lists(*g.neighbor_lists())
    xs = g.position_stars()
    assert _same(xs, m.xs).all()
    for i in range(0, n, max(1, n // 30)):
        xs[i, i % 3] = value
    g.set_position_stars(xs)
    m.xs = xs.copy()
    for name, f in (("compute_densities", m.density), ("compute_pressure_lambdas", m.multipliers),
                    ("compute_pressure_dps", m.dps), ("apply_viscosity", m.viscosity),
                    ("compute_vorticity", m.vorticity), ("apply_vorticity", m.confinement),
                    ("apply_viscosity", m.viscosity), ("compute_densities", m.density),
                    ("compute_pressure_lambdas", m.multipliers), ("compute_pressure_dps", m.dps),
                    ("update_position_stars", m.stars), ("update_velocities", m.velocities)):
        getattr(g, name)()
        f()
        _compare(g, m.state(), name, scratch=True)


@pytest.mark.gpu
@pytest.mark.parametrize("side", [2, 12, 24, 34, 54])
def test_nan_multiplier_at_rest(pbf, scenes, side):
    """Fluid at rest, so that its skin lists serve, and a warm start of zeros
    with one NaN: the NaN moves count as moves, and the skin lists, which leave
    out entries that were 1.1 h away, serve no longer."""
    i = np.arange(side, dtype=F)
    pos = np.stack(np.meshgrid(i, i, i, indexing="ij"), -1).reshape(-1, 3) * F(0.055) + F(0.03)
    n = len(pos)
    vel = np.zeros_like(pos)
    p = _params(pbf, scenes, n, 60, F(0.055) * side + F(0.03))
    g = pbf.Particles(p)
    g.add(pos, pos, vel)
    g.step(2)
    m = Model(p, g.positions(), g.velocities())
    warm = np.zeros(n, F)
    warm[n // 2] = np.nan
    g.set_warm_lambdas(warm)
    g.solve(0.0, 3, pbf.PBF_WARM_GIVEN)
    info = g.solve_info()
    m.forces_predict()
    m.lists(*g.neighbor_lists())
    m.density()
    before = m.xs.copy()
    m.lam = warm
    m.dps()
    m.stars()
    assert np.isnan(m.xs).any()
    for it in range(info["iterations"]):
        m.density()
        m.multipliers()
        if it == 0 and not info["warm_start_kept"]:
            m.xs = before
        elif info["max_error_history"][it] > 0:
            m.dps()
            m.stars()
    m.tail()
    _compare(g, m.state(), "solve")
