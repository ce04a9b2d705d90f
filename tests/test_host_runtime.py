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
