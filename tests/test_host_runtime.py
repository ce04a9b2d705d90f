"""What the library asks of the HIP runtime, on a machine without a GPU: a
stand-in runtime (host_runtime.cpp) records allocations, launches and captured
graphs; no kernel runs.  Each test is a process of its own, with the stand-in
loaded before the library."""
import os
import subprocess
import sys

import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, os, sys
import numpy as np
F = ctypes.CDLL(os.environ["HOST_RUNTIME"], mode=ctypes.RTLD_GLOBAL)
F.fake_set_free.argtypes = [ctypes.c_uint64]
F.fake_launches.argtypes = [ctypes.c_char_p]
F.fake_last_arg.argtypes = [ctypes.c_char_p, ctypes.c_int]
F.fake_last_arg.restype = ctypes.c_uint64
import helpers
from dice_amd import shci, synth
path = os.path.join(os.environ["WORK"], "FCIDUMP")
synth.write_molecular_fcidump(path, 0, 8, 4, 4, 16)
def dets(n, seed):
    return helpers.random_dets(8, 4, 4, n, np.random.default_rng(seed), words=1)
"""


@pytest.fixture(scope="session")
def host_runtime(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rt") / "host_runtime.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", os.path.join(TESTS, "host_runtime.cpp"), "-o", so],
                   check=True)

    def run(script, work, **env):
        e = dict(os.environ, HOST_RUNTIME=so, WORK=str(work), **env)
        e["PYTHONPATH"] = os.pathsep.join([TESTS, os.path.dirname(TESTS), e.get("PYTHONPATH", "")])
        p = subprocess.run([sys.executable, "-c", PRELUDE + script], env=e, stdout=subprocess.PIPE,
                           stderr=subprocess.STDOUT, text=True, timeout=120)
        assert p.returncode == 0, p.stdout

    return run


@pytest.mark.parametrize("change", ["dets", "direct", "precision"])
@pytest.mark.parametrize("storage", ["half", "full"])
def test_graphs_of_a_replaced_hamiltonian_are_not_replayed(storage, change, host_runtime, tmp_path):
    """The block Davidson's captured iterations are replayed while their
    Hamiltonian stands, and never after it was replaced by one of the same
    size: no replayed launch has an argument in freed memory."""
    host_runtime("""
s = shci.System.from_fcidump(path)
opt = dict(davidson_block=True, hip_graphs=True)
def solve():
    s.make_hamiltonian()
    s.davidson(np.eye(5, 1))
    return F.fake_captures()
s.set_options(**opt)
s.set_dets(dets(5, 1))
first = solve()
assert first > 0 and solve() == first  # replayed
change = "%s"
if change == "dets":
    s.set_dets(dets(5, 2))
elif change == "direct":  # without a stored Hamiltonian and back
    s.set_options(direct_sigma=True, **opt)
    solve()
    s.set_options(**opt)
else:
    s.set_options(precision=1, **opt)
    solve()
    s.set_options(**opt)
before = F.fake_captures()
after = solve()
assert F.fake_stale() == 0
assert after == before + first  # captured anew
""" % change, tmp_path, SHCI_STORAGE=storage)


def test_pt_after_a_failed_allocation(host_runtime, tmp_path):
    """Whichever allocation of a PT call fails, the next call on the handle has
    both dense heat-bath tables, filled."""
    host_runtime("""
space = dets(5, 1)
c = np.full(5, 5 ** -0.5)
failed = 0
for k in range(1, 20):
    s = shci.System.from_fcidump(path)
    s.set_dets(space)
    fills = F.fake_launches(b"kDenseHeatBath")
    F.fake_fail_in(k)
    try:
        s.pt_deterministic(c, -1.0, 1e-3)
    except shci.ShciError:
        failed += 1
    F.fake_fail_in(0)
    calls = F.fake_launches(b"kPtGen")
    s.pt_deterministic(c, -1.0, 1e-3)
    assert F.fake_launches(b"kPtGen") > calls
    assert F.fake_last_arg(b"kPtGen", 15) and F.fake_last_arg(b"kPtGen", 16), k  # dense0, dense1
    assert F.fake_launches(b"kDenseHeatBath") >= fills + 2, k
assert failed >= 4  # (the tables, the counts, and what the call itself holds)
""", tmp_path)


def test_full_storage_needs_no_room_for_the_half_forms_order(host_runtime, tmp_path):
    """Full storage takes the tiled copy when its own tables fit.  (No kernel
    runs, so there are no entries: per determinant the inverse permutation,
    x and 64 bytes of slack; per block of 256 rows a segment's tables and
    instruction, offsets and a bitmap of up to 32 tiles.)"""
    host_runtime("""
n = 2000
s = shci.System.from_fcidump(path)
s.set_dets(dets(n, 1))
blocks = (n + 255) // 256
need = n * (4 + 8 + 64) + blocks * (8 + 48) + (blocks + 1) * (24 + 4)
F.fake_set_free(need)
s.make_hamiltonian()
assert F.fake_launches(b"kTileFill") == 1
""", tmp_path, SHCI_STORAGE="full")


@pytest.mark.parametrize("storage,without,held", [
    # what the product reads: entries (2), blockE, the ordered instructions,
    # groups and units; beside them permPos, the sums and their scale
    ("half", {"SHCI_HALF_SIGMA": "rows"}, 9),
    # entries (2), instructions, blockE and blockI, and the segment tables (7),
    # which the next build fills again
    ("full", {"SHCI_SIGMA_LAYOUT": "rows"}, 12)])
def test_tables_of_a_build_are_released(storage, without, held, host_runtime, tmp_path):
    """Buffers that a built Hamiltonian with the tiled copy holds beyond one
    without it."""
    host_runtime("""
def live():
    s = shci.System.from_fcidump(path)
    s.set_dets(dets(50, 1))
    s.make_hamiltonian()
    c = F.fake_live()
    s.close()
    return c
tiled = live()
os.environ.update(%r)
assert F.fake_launches(b"kTileFill") == 1
rows = live()
assert F.fake_launches(b"kTileFill") == 1
assert tiled - rows <= %d, tiled - rows
""" % (without, held), tmp_path, SHCI_STORAGE=storage)
