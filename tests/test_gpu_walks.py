"""GPU tests of the neighbour walks' variants: four lanes per particle in small
scenes, one lane in large ones, over padded lists, skin lists or full lists.
Every variant takes the same pairs and adds them in list order, so all must
equal the CPU oracle bit for bit, on both sides of each size at which the
library changes from one to the other, with list lengths that end inside a
group of four, past a batch of eight and past the 64th entry."""
import os

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

THREADS = max(1, min(16, os.cpu_count() or 1))


def _same(g, o, what):
    s = o.state()
    for name, got in (("x", g.positions()), ("v", g.velocities()), ("rho", g.densities()), ("lam", g.lambdas())):
        assert np.array_equal(got, np.asarray(s[name], dtype=np.float32)), f"{what}: {name}"


def _scene(scenes, counts, squeeze, cap, gamma=0.0):
    """A jittered lattice with its spacing scaled by `squeeze` (denser: longer
    lists and larger corrections) and random velocities."""
    params, pos, vel = scenes.dam_break(counts, tuple(2.0 * c * scenes.SPACING for c in counts), 3, cap=cap, gamma=gamma)
    rng = np.random.default_rng(1)
    vel = rng.uniform(-0.3, 0.3, vel.shape).astype(np.float32)
    return params, (pos * np.float32(squeeze)).astype(np.float32), vel


# (counts, squeeze, cap): particles at, one row past and well past the sizes
# where the walks change: 98,304 and 131,072 and 524,288
SIZES = [((48, 64, 32), 1.0, 60), ((49, 64, 32), 0.84, 128), ((64, 32, 64), 0.84, 128), ((65, 47, 43), 1.0, 47),
         ((128, 64, 64), 1.0, 60), ((81, 81, 81), 0.9, 71)]


@pytest.mark.parametrize("counts,squeeze,cap", SIZES)
def test_fused_step_equals_oracle(pbf, scenes, counts, squeeze, cap):
    params, pos, vel = _scene(scenes, counts, squeeze, cap)
    g = pbf.Particles(params)
    g.add(pos, pos, vel)
    o = O.Oracle(O.params_from_pbf(params), mode=O.JACOBI, threads=THREADS)
    o.set_state(pos, pos, vel)
    g.step(1)
    o.step(1)
    _same(g, o, f"{counts}, squeeze {squeeze}, cap {cap}")
    g.close()


def _passes(g, tension):
    g.apply_external_forces()
    g.predict_positions()
    g.find_neighbors()
    for s in range(4):
        g.compute_densities()
        g.compute_pressure_lambdas()
        g.compute_pressure_dps(substep=s)
        g.update_position_stars()
    g.update_velocities()
    if tension:
        g.apply_surface_tension()
    g.apply_viscosity()
    g.compute_vorticity()
    g.apply_vorticity()
    g.apply_viscosity()
    g.update_positions()


@pytest.mark.parametrize("counts,squeeze,cap", SIZES[:4])
def test_pass_by_pass_equals_oracle(pbf, scenes, counts, squeeze, cap):
    """Two substeps, so that the second list build follows the first one's
    moves (skin lists at rest, full lists where the squeezed block springs
    apart)."""
    params, pos, vel = _scene(scenes, counts, squeeze, cap, gamma=0.5)
    g = pbf.Particles(params)
    g.add(pos, pos, vel)
    o = O.Oracle(O.params_from_pbf(params), mode=O.JACOBI, threads=THREADS)
    o.set_state(pos, pos, vel)
    for _ in range(2):
        _passes(g, True)
    o.step(2)
    _same(g, o, f"{counts}, squeeze {squeeze}, cap {cap}")
    g.close()


def test_pass_lists_after_position_stars_change(pbf, scenes):
    """The per-pass entry points walk the skin lists only while x* is where
    checked moves left it: after positions the caller sets, or a prediction,
    or corrections past the limit, entries outside them may have come within h.
    A context that always walks the full lists gives the same bits."""
    params, pos, vel = _scene(scenes, (20, 17, 19), 1.0, 60)
    rng = np.random.default_rng(5)
    out = []
    for full in (False, True):
        p = params.copy()
        if full:
            p.options |= pbf.PBF_OPT_FULL_LISTS
        g = pbf.Particles(p)
        g.add(pos, pos, vel)
        g.predict_positions()
        g.find_neighbors()
        got = []
        rng = np.random.default_rng(5)
        for how in ("set", "scratch", "predict"):
            shift = rng.uniform(-0.02, 0.02, pos.shape).astype(np.float32)
            if how == "set":
                g.set_position_stars((pos + shift).astype(np.float32))
            elif how == "scratch":  # update_position_stars adds the scratch vector
                g.find_neighbors()
                g.compute_densities()
                g.set_scratch(shift)
                g.update_position_stars()
            else:
                g.find_neighbors()
                g.set_velocities((shift * 100).astype(np.float32))
                g.predict_positions()
            g.compute_densities()
            g.compute_pressure_lambdas()
            g.compute_pressure_dps()
            g.apply_viscosity()
            g.compute_vorticity()
            got += [g.densities(), g.lambdas(), g.scratch(), g.velocities()]
        out.append(got)
        g.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [1, 3, 63, 64, 65, 130])
def test_few_particles(pbf, scenes, n):
    """Quads of a partly filled block, and lists shorter than a group."""
    params, pos, vel = _scene(scenes, (6, 5, 5), 1.0, 60)
    pos, vel = pos[:n].copy(), vel[:n].copy()
    g = pbf.Particles(params)
    g.add(pos, pos, vel)
    o = O.Oracle(O.params_from_pbf(params), mode=O.JACOBI, threads=1)
    o.set_state(pos, pos, vel)
    g.step(2)
    o.step(2)
    _same(g, o, f"{n} particles, fused")
    _passes(g, False)
    o.step(1)
    _same(g, o, f"{n} particles, pass by pass")
    g.close()


@pytest.mark.parametrize("counts", [(11, 9, 10), (49, 46, 44)])
@pytest.mark.parametrize("pairs", [2, 40])
def test_density_fix_next_to_the_walls(pbf, scenes, counts, pairs):
    """Coincident pairs (moved by the density fix) in the corner cells of the
    grid, on its edges and inside, in scenes walked by quads and by single
    lanes: the 5x5x5 cells stamped around a moved particle are cut off at the
    grid's faces, and every particle that lists a moved one is repaired."""
    params, pos, vel = _scene(scenes, counts, 1.0, 60)
    box = np.array(params.boundary_max[:], dtype=np.float32)
    rng = np.random.default_rng(pairs)
    spots = np.stack([rng.choice([0.0, 0.5, 1.0], pairs) for _ in range(3)], axis=1).astype(np.float32)
    lo, hi = pos.min(axis=0), pos.max(axis=0)
    at = lo + spots * (hi - lo)
    ids = rng.permutation(len(pos))[:2 * pairs]
    pos[ids] = np.repeat(np.clip(at, 0.0, box), 2, axis=0)
    vel[ids] = np.repeat(rng.uniform(-0.2, 0.2, (pairs, 3)), 2, axis=0).astype(np.float32)
    g = pbf.Particles(params)
    g.add(pos, pos, vel)
    o = O.Oracle(O.params_from_pbf(params), mode=O.JACOBI, threads=THREADS)
    o.set_state(pos, pos, vel)
    g.step(1)
    o.step(1)
    assert g.stats()["density_hacks"] > 0
    _same(g, o, f"{pairs} pairs, {len(pos)} particles")
    g.close()


# at and past the sizes where sixteen lanes give way to four (12,288 particles
# in the pressure solve, 24,576 after it), with lists that end inside a step of
# sixteen, within its first eight and past the 64th entry
@pytest.mark.parametrize("counts,squeeze,cap", [((1, 1, 1), 1.0, 60), ((5, 4, 3), 0.84, 128), ((9, 9, 9), 1.0, 17),
                                                ((24, 16, 32), 0.84, 128), ((1, 12289, 1), 0.9, 60),
                                                ((32, 24, 32), 0.9, 71), ((24, 32, 33), 1.0, 41)])
def test_sixteen_lanes_equal_oracle(pbf, scenes, counts, squeeze, cap):
    params, pos, vel = _scene(scenes, counts, squeeze, cap)
    g = pbf.Particles(params)
    g.add(pos, pos, vel)
    o = O.Oracle(O.params_from_pbf(params), mode=O.JACOBI, threads=THREADS)
    o.set_state(pos, pos, vel)
    for k in range(3):  # (the later steps over skin lists, where no particle moves far)
        g.step(1)
        o.step(1)
        _same(g, o, f"{counts}, squeeze {squeeze}, cap {cap}, step {k + 1}")
    g.close()


@pytest.mark.parametrize("counts", [(10, 9, 8), (50, 53, 50)])
def test_tension_after_a_partial_color_pass(pbf, scenes, counts):
    """Surface tension takes a neighbour's density from the color pass when
    that ran over every particle in the same call, and from the densities
    otherwise: the color field in two halves, the second with the forces, must
    give what one call gives (four lanes and one lane a particle)."""
    params, pos, vel = _scene(scenes, counts, 0.9, 60, gamma=0.5)
    n = pos.shape[0]
    out = []
    for halves in (False, True):
        g = pbf.Particles(params)
        g.add(pos, pos, vel)
        g.find_neighbors()
        g.compute_densities()
        g.set_scratch(np.full_like(pos, 7.0))  # (no color left from before)
        if halves:
            g.apply_surface_tension(pbf.span(0, n // 2), pbf.span(0, 0))
            g.apply_surface_tension(pbf.span(n // 2, n), pbf.span(0, n))
        else:
            g.apply_surface_tension()
        out.append((g.scratch(), g.velocities()))
        g.close()
    assert not np.array_equal(out[0][1], vel)
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("counts,squeeze,cap", [((64, 48, 48), 0.84, 128), ((73, 45, 45), 0.9, 71)])
def test_density_by_lanes_and_update_by_quads(pbf, scenes, counts, squeeze, cap):
    """At 147,456 particles (and one row more) the density pass goes by single
    lanes and the pressure update by quads (by single lanes)."""
    params, pos, vel = _scene(scenes, counts, squeeze, cap)
    g = pbf.Particles(params)
    g.add(pos, pos, vel)
    o = O.Oracle(O.params_from_pbf(params), mode=O.JACOBI, threads=THREADS)
    o.set_state(pos, pos, vel)
    g.step(1)
    o.step(1)
    _same(g, o, f"{counts}, squeeze {squeeze}, cap {cap}")
    g.close()
