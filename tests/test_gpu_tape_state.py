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


# (steps, checkpoint interval): again the same, fewer in what the last one held, more, one set of segment
# buffers after two, none re-run after some
TAPES = [(8, 4), (8, 4), (3, 4), (12, 2), (12, 2), (1, 1), (8, 4), (2, 8)]


def _fresh_gradients(probs, seeds, steps, every):
    from cumpic_amd.cumc import Batch, Solver
    solvers = [Solver.from_problem(p) for p in probs]
    b = Batch(solvers)
    b.tape_run(steps, every)
    return b.tape_backward(seeds)


def test_gradients_do_not_depend_on_earlier_tapes():
    """Memory kept from one tape to the next: every gradient is a fresh object's bit for bit, for one box and
    for a batch, and for a box used alone between two batch tapes."""
    from cumpic_amd.cumc import Batch, Solver
    probs = [_box(16, 6), _box(24, 7)]
    seeds = _seeds(probs)
    solvers = [Solver.from_problem(p) for p in probs]
    b = Batch(solvers)
    for steps, every in TAPES:
        want = _fresh_gradients(probs, seeds, steps, every)
        one = Solver.from_problem(probs[1])
        one.tape_run(steps, every)
        alone = one.tape_backward(seed_bcell=seeds[1])[0]
        for s, p in zip(solvers, probs):
            s.upload(p.prim, p.eps)
        b.tape_run(steps, every)
        for i, g in enumerate(b.tape_backward(seeds)):
            assert np.array_equal(g, want[i]), f"batch, {steps} steps every {every}, box {i}"
        solvers[1].upload(probs[1].prim, probs[1].eps)
        solvers[1].tape_run(steps, every)
        assert np.array_equal(solvers[1].tape_backward(seed_bcell=seeds[1])[0], alone), f"alone, {steps} every {every}"


def _free_bytes():
    import ctypes
    from cumpic_amd.cumc import lib
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_a_small_tape_gives_a_large_one_back():
    """A tape holds what it needs: device memory after a small tape does not depend on one before it."""
    from cumpic_amd.cumc import Solver
    s = Solver.from_problem(_box(256, 8))
    s.tape_run(1, 1)
    free = _free_bytes()
    s.tape_run(4, 4)  # about 1.7 times the states
    s.tape_run(1, 1)
    assert _free_bytes() >= free - (8 << 20)
