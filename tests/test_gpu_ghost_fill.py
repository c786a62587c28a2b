"""The one-launch ghost fill against the restatement's three passes, every ghost entry bit for bit.

Every boundary kind on every side, also different kinds on the two sides of an axis (where the y-outer
side's eps follows its own rule, or is left as it was), on boxes down to one cell along an axis, from
arrays whose ghost entries hold other values than the fill leaves.
"""
import dataclasses

import numpy as np
import pytest

from cumpic_amd.config import MODEL_TORUS_CYN, MODEL_TORUS_SPH, Config, uniform_faces
from tests.helpers import assert_bitwise

pytestmark = pytest.mark.gpu

FLAGS = [(0,) * 6, (1,) * 6, (2,) * 6, (3, 3, 3, 3, 2, 2), (2, 1, 4, 4, 4, 4), (1, 0, 0, 1, 1, 0), (0, 1, 1, 0, 0, 1),
         (2, 0, 2, 0, 0, 2), (1, 2, 0, 2, 2, 0), (3, 1, 1, 3, 1, 4), (0, 0, 1, 2, 0, 0), (1, 1, 2, 1, 1, 1)]


def _random(flags, shape, model=0):
    from cumpic_amd.ics import Problem
    nx, ny, nz = shape
    cfg = Config(nx=nx, ny=ny, nz=nz, boundary_flag=flags, cfl=0.3)
    if model:
        cfg = dataclasses.replace(cfg, model=model, coordinate=2, rho_floor=1e-4, eps_floor=1e-6, r_sh=0.5)
    rng = np.random.default_rng(hash((flags, shape)) % 2**32)
    prim = rng.uniform(-0.5, 0.5, cfg.shape + (8,))
    prim[..., 0] = rng.uniform(0.5, 1.5, cfg.shape)
    prim[..., 4] = rng.uniform(0.5, 1.5, cfg.shape)
    eps = rng.uniform(0.5, 1.5, cfg.shape)
    return Problem(cfg, uniform_faces(nx, 1.0, 2.0) + (0.5 if model else 0.0), uniform_faces(ny, 0.0, 1.0), uniform_faces(nz, 0.0, 1.0), prim, eps)


@pytest.mark.parametrize("shape", [(7, 5, 4), (3, 3, 3), (12, 3, 1), (1, 1, 1), (70, 1, 3)])
@pytest.mark.parametrize("flags", FLAGS)
def test_fill_matches_three_passes(flags, shape):
    if any(f >= 2 and shape[s // 2] < 3 for s, f in enumerate(flags)):
        pytest.skip("parity copies need three interior cells")
    _check(_random(flags, shape))


@pytest.mark.parametrize("flags", [(1, 1, 0, 0, 1, 1), (2, 1, 0, 0, 2, 1)])
def test_fill_with_inflow_clamps(flags):
    _check(_random(flags, (9, 6, 8), model=MODEL_TORUS_CYN))


def _check(prob):
    from cumpic_amd.cumc import Solver
    from oracle.oracle import Oracle
    g, o = Solver.from_problem(prob), Oracle.from_problem(prob)
    g.initial_update()
    o.initial_update()
    for step in range(2):
        a, b = g.download(), o.get_state()
        for k in ("prim", "eps", "bcell"):
            assert_bitwise(a[k], b[k], f"{k}, step {step}")
        g.rungekutta(1.0e-4)
        o.rungekutta(1.0e-4)


@pytest.mark.parametrize("flags", [(1, 1, 1, 1, 0, 0), (2, 1, 1, 2, 0, 0), (1, 2, 0, 0, 1, 1)])
def test_fill_with_spherical_inflow_clamps(flags):
    """r ghosts take no inflow; the z ones (phi) are as the boundary leaves them."""
    p = _random(flags, (9, 6, 8), model=MODEL_TORUS_CYN)
    cfg = dataclasses.replace(p.cfg, model=MODEL_TORUS_SPH, coordinate=3, r_sh=0.1)
    _check(dataclasses.replace(p, cfg=cfg, xf=uniform_faces(9, 2.0, 3.0), yf=uniform_faces(6, 1.2, 1.9), zf=uniform_faces(8, 0.0, 1.0)))


@pytest.mark.parametrize("shape", [(7, 5, 4), (3, 3, 3), (12, 3, 1), (70, 1, 3)])
@pytest.mark.parametrize("flags", FLAGS)
def test_fp32_fill_matches_fp64_fill(flags, shape):
    """Mixed form: fluxes over the FP32 planes whose ghosts a step's own fill left, against those of a context
    that takes the same state and fills in FP64.  Bit for bit, but where a y-outer ghost's eps does not come
    from its density's cell: there the pressure is formed from rounded factors (2^-24 each and one rounding),
    which a face flux of either side's states carries with a factor of order one."""
    from cumpic_amd.config import MIXED
    from cumpic_amd.cumc import Solver
    if any(f >= 2 and shape[s // 2] < 3 for s, f in enumerate(flags)):
        pytest.skip("parity copies need three interior cells")
    prob = _random(flags, shape)
    s = Solver.from_problem(prob, precision=MIXED)
    s.initial_update()
    s.rungekutta(1.0e-4)
    got = [s.sweep_flux(d) for d in (1, 2, 3)]
    state = s.download()
    t = Solver.from_problem(prob, precision=MIXED)
    t.upload(state["prim"], state["eps"])
    t.initial_update()
    own_rule = (flags[2] == 0) != (flags[3] == 0)
    for d in (1, 2, 3):
        want = t.sweep_flux(d)
        if own_rule:
            assert np.max(np.abs(got[d - 1] - want)) <= 16 * 2.0**-24 * np.max(np.abs(want)), f"flux {d}"
        else:
            assert_bitwise(got[d - 1], want, f"flux {d}")
