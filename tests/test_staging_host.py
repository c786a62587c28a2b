"""The staged transfers' units, waits and errors over a stand-in for the HIP runtime, on the CPU."""
import ctypes
import os
import subprocess

import pytest

from cumpic_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "native", "staging_host.hip")
OUT = os.path.join(HERE, "native", "_build", "libstaging_host.so")
CSRC = os.path.join(HERE, "..", "cumpic_amd", "csrc")


@pytest.fixture(scope="module")
def built():
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    deps = [SRC] + [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hpp") or f == "cumc_transfer.hip"]
    if not os.path.exists(OUT) or os.path.getmtime(OUT) < max(map(os.path.getmtime, deps)):
        obj = OUT + ".o"
        # linked without the HIP runtime: the file defines the calls it makes
        for cmd in ([build.HIPCC, *build.COMMON, "-O1", "-w", "-c", "-o", obj, SRC],
                    ["g++", "-shared", "-o", OUT + ".tmp", obj, "-Wl,-Bsymbolic", "-lpthread"]):
            r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
            assert r.returncode == 0, r.stdout
        os.replace(OUT + ".tmp", OUT)
    return OUT


@pytest.fixture
def stg(built, tmp_path):
    # a copy of its own for each test: the library keeps its units in static storage
    path = str(tmp_path / "libstaging_host.so")
    with open(built, "rb") as f, open(path, "wb") as g:
        g.write(f.read())
    L = ctypes.CDLL(path)
    L.stg_allow.argtypes = [ctypes.c_long, ctypes.c_long]
    for f in ("stg_streams_made", "stg_allocs_made", "stg_live"):
        getattr(L, f).restype = ctypes.c_long
    L.stg_retain()
    return L


MANY = 1 << 40
SMALL, LARGE = (3, 4, 2), (70, 64, 60)  # one unit, room for eight


@pytest.mark.parametrize("shape", [SMALL, (26, 26, 26), (27, 26, 26), (300, 1, 1), LARGE])
def test_round_trip(stg, shape):
    assert stg.stg_round_trip(*shape) == 0
    assert stg.stg_round_trip(*shape) == 0
    assert stg.stg_unfinished() == 0
    stg.stg_release()
    assert stg.stg_live() == 0


def test_goes_on_with_the_units_it_has_when_memory_is_short(stg):
    """A unit that cannot be made leaves a transfer to those there are, and no error behind."""
    assert stg.stg_round_trip(*SMALL) == 0
    stg.stg_allow(0, MANY)
    assert stg.stg_round_trip(*LARGE) == 0
    assert stg.stg_round_trip(*LARGE) == 0
    stg.stg_allow(MANY, MANY)
    assert stg.stg_round_trip(*LARGE) == 0


def test_first_unit_refused_is_an_error_and_not_the_last_word(stg):
    stg.stg_allow(0, MANY)
    assert stg.stg_round_trip(*SMALL) == 10 + 4  # CUMC_ENOMEM
    stg.stg_allow(MANY, MANY)
    assert stg.stg_round_trip(*SMALL) == 0


@pytest.mark.parametrize("shape", [SMALL, LARGE])
@pytest.mark.parametrize("launches", [0, 1, 5])
def test_failed_piece_leaves_no_work_behind(stg, shape, launches):
    """A transfer that fails waits for what it queued: its buffers go to the next transfer."""
    assert stg.stg_round_trip(*shape) == 0
    stg.stg_allow(MANY, launches)
    assert stg.stg_round_trip(*shape) == (10 + 2 if shape == LARGE or launches < 4 else 0)
    assert stg.stg_unfinished() == 0
    stg.stg_allow(MANY, MANY)
    assert stg.stg_round_trip(*shape) == 0


def test_units_and_streams_are_made_as_transfers_earn_them(stg):
    """A process that opens one context at a time pays little for units it will hardly use; one that
    transfers again and again has all of them soon."""
    assert stg.stg_round_trip(*SMALL) == 0
    assert (stg.stg_streams_made(), stg.stg_allocs_made()) == (1, 2)  # the context's own stream
    stg.stg_release()
    stg.stg_retain()
    streams, allocs = stg.stg_streams_made(), stg.stg_allocs_made()
    assert stg.stg_round_trip(*LARGE) == 0
    assert stg.stg_streams_made() - streams <= 3 and stg.stg_allocs_made() - allocs == 2
    for _ in range(20):
        assert stg.stg_round_trip(*LARGE) == 0
    assert stg.stg_streams_made() - streams == 7 and stg.stg_allocs_made() - allocs == 2
    stg.stg_release()
    assert stg.stg_live() == 0
