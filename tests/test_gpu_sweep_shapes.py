"""The sweeps' launch shapes: pencil segments chosen by the grid's size, and the wave-parallel y sweep.

Whatever shape a grid takes, its step is the CPU restatement's bit for bit.  The grids lie on both
sides of the choices: a few wavefronts (segments of one face), one to several wavefronts per compute
unit, segments that do not divide the pencil, pencils shorter than a segment, and flat boxes.
"""
import numpy as np
import pytest

from cumpic_amd import ics
from tests.helpers import assert_bitwise

pytestmark = pytest.mark.gpu

GRIDS = [(5, 4, 3), (16, 16, 16), (37, 23, 29), (64, 12, 31), (20, 130, 6), (9, 8, 140), (70, 66, 50), (150, 17, 1), (31, 200, 1)]


def _problem(grid, recon):
    nx, ny, nz = grid
    p = ics.spectral_box(n=max(nx, ny, nz), seed=21, v_rms=0.3, db_rms=0.3, ndim=2 if nz == 1 else 3)
    c = p.cfg
    c.nx, c.ny, c.nz, c.recon = nx, ny, nz, recon
    c.boundary_flag = (1,) * 6
    p.xf, p.yf, p.zf = p.xf[:nx + 7].copy(), p.yf[:ny + 7].copy(), p.zf[:nz + 7].copy()
    p.prim = np.ascontiguousarray(p.prim[:nz + 6, :ny + 6, :nx + 6])
    p.eps = np.ascontiguousarray(p.eps[:nz + 6, :ny + 6, :nx + 6])
    return ics.randomize(p, seed=3, amp=0.1)


@pytest.mark.parametrize("recon", [4, 1])
@pytest.mark.parametrize("grid", GRIDS)
def test_step_matches_restatement(grid, recon):
    from cumpic_amd.cumc import Solver
    from oracle.oracle import Oracle
    prob = _problem(grid, recon)
    g, o = Solver.from_problem(prob), Oracle.from_problem(prob)
    g.initial_update()
    o.initial_update()
    for _ in range(2):
        dt = g.finddt()
        assert dt == o.finddt()
        g.rungekutta(dt)
        o.rungekutta(dt)
    a, b = g.download(), o.get_state()
    for k in ("prim", "eps", "bcell"):
        assert_bitwise(a[k], b[k], k)


# states whose quotients leave the range of the shared reciprocals in part of the box (fields below
# 2^-300, densities and pressures below 2^-300 or above 2^300, zeros of both signs), so that a
# wavefront takes both forms of the FP64 face
EXTREMES = {
    "tiny_b": lambda p, s: _scale(p, s, (5, 6, 7), 1e-95),
    "subnormal_b": lambda p, s: _scale(p, s, (5, 6, 7), 1e-158),
    "tiny_v": lambda p, s: _scale(p, s, (1, 2, 3), 1e-200),
    "zero_v_and_b": lambda p, s: _scale(p, s, (1, 2, 3, 5, 6, 7), -0.0),
    "tiny_rho_p": lambda p, s: _scale(p, s, (0, 4), 1e-95),
    "huge_rho_p": lambda p, s: _scale(p, s, (0, 4), 1e95),
    "zero_p": lambda p, s: _scale(p, s, (4,), 0.0),
    "huge_b": lambda p, s: _scale(p, s, (5, 6, 7), 1e70),
}


def _scale(p, where, comps, factor):
    for c in comps:
        p.prim[where + (c,)] *= factor


@pytest.mark.parametrize("recon", [4, 1])
@pytest.mark.parametrize("kind", sorted(EXTREMES))
def test_extreme_states_match_restatement(kind, recon):
    from cumpic_amd.cumc import Solver
    from oracle.oracle import Oracle
    prob = _problem((21, 19, 17), recon)
    EXTREMES[kind](prob, (slice(6, 14), slice(5, 15), slice(7, 17)))
    prob.eps[...] = prob.prim[..., 4] / prob.prim[..., 0] / (prob.cfg.ggas - 1.0)
    g, o = Solver.from_problem(prob), Oracle.from_problem(prob)
    g.initial_update()
    o.initial_update()
    for d in (1, 2, 3):
        a, b = g.sweep_flux(d), o.sweep_flux(d)
        n = (prob.cfg.nx, prob.cfg.ny, prob.cfg.nz)
        sl = tuple(slice(2, 3 + n[ax] + (ax + 1 != d)) for ax in (2, 1, 0))
        assert_bitwise(a[sl], b[sl], f"{kind}: flux {d}")
    dt = g.finddt()
    assert dt == o.finddt()
    g.rungekutta(dt)
    o.rungekutta(dt)
    a, b = g.download(), o.get_state()
    for k in ("prim", "eps", "bcell"):
        assert_bitwise(a[k], b[k], f"{kind}: {k}")


@pytest.mark.parametrize("grid", [(7, 5, 1), (21, 18, 13), (130, 40, 33)])
def test_one_launch_matches_separate_sweeps(grid):
    """Sweeps timed one by one (profiling on) and in one launch give the same step."""
    from cumpic_amd.cumc import Solver
    states = []
    for on in (False, True):
        g = Solver.from_problem(_problem(grid, 4))
        g.initial_update()
        g.profile(on)
        g.run(3)
        states.append(g.download())
        g.close()
    for k in ("prim", "eps", "bcell"):
        assert_bitwise(states[0][k], states[1][k], k)


# a few long pencils along y: the wave-parallel y sweep beside the joined one, and grids just short of it;
# one plane (z-collapsed) and the three planes of a box that is not
@pytest.mark.parametrize("recon", [4, 1])
@pytest.mark.parametrize("nx,ny,collapse", [(1, 4096, True), (2, 4200, True), (10, 4160, True), (11, 4160, True), (1, 4095, True),
                                            (2, 12288, False), (3, 12288, False)])
def test_long_thin_grids_match_restatement(nx, ny, collapse, recon):
    from cumpic_amd.config import Config, uniform_faces
    from cumpic_amd.cumc import Solver
    from cumpic_amd.ics import Problem
    from oracle.oracle import Oracle
    cfg = Config(nx=nx, ny=ny, nz=1, boundary_flag=(1,) * 6, recon=recon, cfl=0.3)
    rng = np.random.default_rng(7)
    prim = rng.uniform(-0.2, 0.2, cfg.shape + (8,))
    prim[..., 0], prim[..., 4] = rng.uniform(0.5, 1.5, cfg.shape), rng.uniform(0.5, 1.5, cfg.shape)
    prob = Problem(cfg, uniform_faces(nx, 0.0, 1.0), uniform_faces(ny, 0.0, 64.0), uniform_faces(1, 0.0, 1.0), prim,
                   prim[..., 4] / prim[..., 0] / (cfg.ggas - 1.0))
    g, o = Solver.from_problem(prob), Oracle.from_problem(prob)
    g.set_zcollapse(collapse)
    g.initial_update()
    o.initial_update()
    for _ in range(2):
        dt = g.finddt()
        assert dt == o.finddt()
        g.rungekutta(dt)
        o.rungekutta(dt)
    a, b = g.download(), o.get_state()
    for k in ("prim", "eps", "bcell"):
        assert_bitwise(a[k], b[k], k)
