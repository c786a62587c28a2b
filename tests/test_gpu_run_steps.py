"""Steps of one run, which hand the time step on by themselves, against steps called one by one."""
import os
import subprocess
import sys

import numpy as np
import pytest

from cumpic_amd import ics
from cumpic_amd.config import FP64, MIXED
from tests.helpers import assert_bitwise

pytestmark = pytest.mark.gpu

ROOT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..")

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


@pytest.mark.parametrize("mixed", [False, True])
def test_profile_counts_the_launches_it_says(mixed):
    from cumpic_amd.config import FP64, MIXED
    from cumpic_amd.cumc import Solver
    s = Solver.from_problem(ics.spectral_box(n=20, seed=3), precision=MIXED if mixed else FP64)
    s.initial_update()
    sweeps = ("flux_x", "flux_y", "flux_z", "flux_xyz")
    for joined in (False, True):
        s.profile(True, joined=joined)
        s.run(2)
        n = {k: v[1] for k, v in s.kernel_times().items()}
        assert [n[k] for k in sweeps] == ([0, 0, 0, 6] if joined and not mixed else [6, 6, 6, 0])
        assert n["tail"] == n["ecorn"] == n["ghost"] == 6


def test_tuner_leaves_values_that_change_no_launch():
    """On a small grid every segment length and plane chunk comes to one face and one plane: nothing to choose."""
    from cumpic_amd.cumc import Batch, Solver
    solvers = [Solver.from_problem(ics.small_periodic(8)) for _ in range(2)]
    for s in solvers:
        s.initial_update()
    solvers[0].set_tuning({**solvers[0].tuning(), "seg": 17, "zchunk": 5})
    t = solvers[0].autotune()
    assert (t["seg"], t["zchunk"]) == (17, 5)
    b = Batch(solvers)
    seg = b.tuning()["seg"]
    assert b.autotune()["seg"] == (seg if seg > 0 else 24)


BLOCKING = """
import time
from cumpic_amd import ics
from cumpic_amd.cumc import Solver, lib
assert lib().hipSetDeviceFlags(4) == 0  # hipDeviceScheduleBlockingSync
s = Solver.from_problem(ics.spectral_box(n=128))
s.initial_update()
s.run(20)
wall, cpu = time.perf_counter(), time.process_time()
s.run(100)
print(time.process_time() - cpu, time.perf_counter() - wall)
"""


def test_run_waits_as_the_device_is_set_to():
    """With blocking waits chosen, a run's steps leave the core to others (watching takes all of it)."""
    out = subprocess.run([sys.executable, "-c", BLOCKING], cwd=ROOT, stdout=subprocess.PIPE, text=True, timeout=100)
    assert out.returncode == 0
    cpu, wall = (float(v) for v in out.stdout.split())
    assert cpu < 0.75 * wall
