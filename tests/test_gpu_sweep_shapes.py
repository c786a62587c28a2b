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
