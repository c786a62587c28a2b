"""A backward pass reverses a tape that was recorded to its end, or is refused."""
import numpy as np
import pytest

from cumpic_amd import ics

pytestmark = pytest.mark.gpu


def _box(n, seed):
    return ics.randomize(ics.spectral_box(n=n, ndim=2, seed=seed), seed=seed, amp=0.05)


def _seeds(probs):
    return [np.random.default_rng(5).standard_normal(p.cfg.shape + (3,)) for p in probs]


def _refused(call, what="must precede"):
    from cumpic_amd.cumc import CumcError
    with pytest.raises(CumcError, match=what):
        call()


@pytest.mark.parametrize("every", [8, 2])
def test_failed_batch_tape_is_not_reversed(every):
    from cumpic_amd.cumc import Batch, Solver
    probs = [_box(16, 1), _box(20, 2)]
    seeds = _seeds(probs)
    solvers = [Solver.from_problem(p) for p in probs]
    b = Batch(solvers)
    _refused(lambda: b.tape_backward(seeds))
    b.tape_run(5, every)
    want = b.tape_backward(seeds)
    nan = probs[1].prim.copy()
    nan[3, 9, 9, 0] = np.nan
    solvers[1].upload(nan, probs[1].eps)
    solvers[0].upload(probs[0].prim, probs[0].eps)
    _refused(lambda: b.tape_run(5, every), "non-finite")
    _refused(lambda: b.tape_backward(seeds))
    for s, p in zip(solvers, probs):
        s.upload(p.prim, p.eps)
    b.tape_run(5, every)
    for g, w in zip(b.tape_backward(seeds), want):
        assert np.array_equal(g, w)


def test_failed_tape_is_not_reversed():
    from cumpic_amd.cumc import Solver
    p = _box(16, 3)
    seed = _seeds([p])[0]
    s = Solver.from_problem(p)
    dts = s.tape_run(4, 2)
    want = s.tape_backward(seed_bcell=seed)
    s.upload(p.prim, p.eps)
    _refused(lambda: s.tape_run(4, 2, dts=np.array([dts[0], np.nan, dts[2], dts[3]])), "frozen dt")
    _refused(lambda: s.tape_backward(seed_bcell=seed))
    s.upload(p.prim, p.eps)
    s.tape_run(4, 2)
    for g, w in zip(s.tape_backward(seed_bcell=seed), want):
        assert np.array_equal(g, w)


def test_a_box_holds_one_tape():
    """A box taped by itself leaves the batch's tape, and the other way round."""
    from cumpic_amd.cumc import Batch, Solver
    probs = [_box(16, 4), _box(20, 5)]
    seeds = _seeds(probs)
    solvers = [Solver.from_problem(p) for p in probs]
    b = Batch(solvers)
    b.tape_run(5, 2)
    _refused(lambda: solvers[0].tape_backward(seed_bcell=seeds[0]))
    solvers[0].upload(probs[0].prim, probs[0].eps)
    solvers[0].tape_run(3, 8)
    _refused(lambda: b.tape_backward(seeds))
    solvers[0].tape_backward(seed_bcell=seeds[0])
    solvers[0].tape_free()
    _refused(lambda: b.tape_backward(seeds))
    _refused(lambda: solvers[0].tape_backward(seed_bcell=seeds[0]))
