"""Staged host transfers: what is uploaded comes back, at the ends of the pieces and from several threads."""
import threading

import numpy as np
import pytest

from cumpic_amd.config import Config, uniform_faces

pytestmark = pytest.mark.gpu


def _solver(shape):
    from cumpic_amd.cumc import Solver
    nx, ny, nz = shape
    return Solver(Config(nx=nx, ny=ny, nz=nz), uniform_faces(nx, 0.0, 1.0), uniform_faces(ny, 0.0, 1.0), uniform_faces(nz, 0.0, 1.0))


def _round_trip(s, seed):
    rng = np.random.default_rng(seed)
    prim, eps = rng.standard_normal(s.cfg.shape + (8,)), rng.standard_normal(s.cfg.shape)
    s.upload(prim, eps)
    d = s.download()
    return np.array_equal(d["prim"], prim) and np.array_equal(d["eps"], eps) and not d["bcell"].any()


# a piece holds 32768 cells of prim, 262144 of eps: one cell, exactly one piece, one row more, several
# pieces and threads, a plane wider than a piece
@pytest.mark.parametrize("shape", [(1, 1, 1), (26, 26, 26), (27, 26, 26), (58, 58, 58), (59, 58, 58), (40000, 1, 1), (90, 70, 50)])
def test_round_trip(shape):
    s = _solver(shape)
    assert _round_trip(s, 1) and _round_trip(s, 2)


def test_round_trip_from_threads():
    ok = []
    solvers = [_solver((40 + 3 * i, 33, 20 + i)) for i in range(10)]
    threads = [threading.Thread(target=lambda s=s, i=i: ok.extend(_round_trip(s, 10 * i + r) for r in range(4))) for i, s in enumerate(solvers)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert ok == [True] * 40
