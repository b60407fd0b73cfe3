"""The library builds without the tests' sources, and the register tile gives the
same bits on a team that offers only the basic interface (one slot per wave, no
best_slot), as the CPU harness of an earlier tree has it."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def bare(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("bare") / "libbare.so")
    subprocess.check_call(["g++", "-O1", "-ffp-contract=off", "-fno-fast-math", "-fPIC", "-std=c++20", "-pthread",
                           "-I" + os.path.join(ROOT, "tensorcrossinterpolation.jl_amd", "csrc"),
                           "-I" + os.path.join(ROOT, "include"), "-shared", "-o", out,
                           os.path.join(HERE, "engine_host", "bare_team.cpp")])
    lib = C.CDLL(out)
    dp, ip = C.POINTER(C.c_double), C.POINTER(C.c_int32)
    lib.eh_rrlu_bare.argtypes = [dp, C.c_int, C.c_int, C.c_int64, C.c_double, C.c_double, C.c_int, ip, ip, dp]
    return lib


@pytest.mark.parametrize("m,n,lo", [(1, 1, 1), (64, 4, 0), (65, 31, 1), (20, 128, 0), (128, 128, 1)])
def test_bare_team(bare, m, n, lo):
    rng = np.random.default_rng(7 * m + n)
    # few values, so that the search has ties within a wave and between waves
    A = np.asfortranarray(rng.integers(-3, 4, (m, 5)) @ rng.integers(-3, 4, (5, n)) * 0.25)
    A += np.asfortranarray(1e-9 * rng.standard_normal((m, n)))
    A[0, 0] = A[m - 1, n - 1] = 50.0
    rp, cp, err = np.zeros(m, np.int32), np.zeros(n, np.int32), C.c_double()
    dp, ip = C.POINTER(C.c_double), C.POINTER(C.c_int32)
    p = bare.eh_rrlu_bare(A.ctypes.data_as(dp), m, n, 1 << 40, 1e-6, 0.0, lo, rp.ctypes.data_as(ip),
                          cp.ctypes.data_as(ip), C.byref(err))
    o = O.rrlu(A, reltol=1e-6, leftorthogonal=bool(lo))
    assert p == o.npivot
    assert np.array_equal(rp + 1, o.rowpermutation) and np.array_equal(cp + 1, o.colpermutation)
    assert err.value == o.error


@pytest.mark.parametrize("harness", [0, 2])
def test_build_without_the_harness(tmp_path, harness):
    """build() with a `make` that only reports its directory and fails for the tests'."""
    mk = tmp_path / "make"
    mk.write_text("#!/bin/sh\nfor d; do :; done\necho \"made $d\"\ncase \"$d\" in */tests/engine_host) exit %d;; esac\n"
                  % harness)
    mk.chmod(0o755)
    code = ("import sys; sys.path.insert(0, %r); import os, __graft_entry__ as g; os.remove = lambda p: print('removed', p)\n"
            "g.build(); print('built')" % ROOT)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                       env=dict(os.environ, PATH=f"{tmp_path}:{os.environ['PATH']}"))
    assert r.returncode == 0, r.stderr
    assert "csrc" in r.stdout and "engine_host" in r.stdout and r.stdout.rstrip().endswith("built")
    assert ("did not compile" in r.stderr) == (harness != 0)
