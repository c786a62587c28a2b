"""Steps of one run, which hand the time step on by themselves, against steps called one by one."""
import numpy as np
import pytest

from cumpic_amd import ics
from cumpic_amd.config import FP64, MIXED
from tests.helpers import assert_bitwise

pytestmark = pytest.mark.gpu

PROBLEMS = {
    "box": lambda: ics.randomize(ics.small_periodic(17, seed=5), seed=6, amp=0.1),
    "flat": lambda: ics.spectral_box(n=40, seed=7, ndim=2),
    "torus": lambda: ics.torus_cyn(nr=20, nphi=8, nzz=18),
}


def _start(name, precision):
    from cumpic_amd.cumc import Solver
    s = Solver.from_problem(PROBLEMS[name](), precision=precision)
    s.initial_update()
    return s


@pytest.mark.parametrize("steps", [3, 11])  # direct launches; step graphs
@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("name", sorted(PROBLEMS))
def test_run_matches_single_steps(name, precision, steps):
    a, b = _start(name, precision), _start(name, precision)
    t, dts = 0.0, []
    for _ in range(steps):
        dt = b.finddt()
        b.rungekutta(dt)
        dts.append(dt)
        t += dt
    # ended by the step count, then by the time (the last step cut short)
    got, tg = a.run(steps)
    assert_bitwise(got, np.array(dts), "dt")
    assert tg == t
    dt = b.finddt()
    end = t + 1.5 * dt
    got, tg = a.run(steps, total_time=end, t0=t)
    b.rungekutta(dt)
    last = end - (t + dt)
    b.rungekutta(last)
    assert_bitwise(got, np.array([dt, last]), "cut dt")
    assert tg == t + dt + last
    x, y = a.download(), b.download()
    for k in ("prim", "eps", "bcell"):
        assert_bitwise(x[k], y[k], k)


def test_run_stops_at_a_non_finite_step():
    from cumpic_amd.cumc import CumcError, Solver
    p = PROBLEMS["box"]()
    good = p.prim.copy()
    p.prim[9, 9, 9, 1] = 1.0e200  # its square overflows in the first step
    s = Solver.from_problem(p)
    s.initial_update()
    with pytest.raises(CumcError, match="non-finite"):
        s.run(12)
    p.prim[...] = good
    s.upload(p.prim, p.eps)
    s.initial_update()
    fresh = _start("box", FP64)
    assert_bitwise(s.run(9)[0], fresh.run(9)[0], "dt after the error")
