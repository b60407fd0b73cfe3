"""Results of a batch read through tci_batch_solution and through the
per-set and per-tensor accessors: the same values whatever is asked first,
for one solve or many, for solves of different length in one batch, with and
without a history, and for solves that ended with an error."""
import ctypes as C

import numpy as np
import pytest

from problems import specs
from test_gpu_solves import _check, _tci_problem

pytestmark = pytest.mark.gpu


def _submit(tci, ctx, problems):
    lib = tci._abi.lib()
    hs = [tci._holder(*p) for p in problems]
    arr = (tci._abi.tci_problem * len(hs))(*[h.st for h in hs])
    b = C.c_void_p()
    assert lib.tci_solve_submit(ctx.handle, len(hs), arr, C.byref(b)) == 0
    assert lib.tci_batch_wait(b) == 0
    return b


def _sets(tci, b, i, L):
    lib, out = tci._abi.lib(), []
    for which in range(4):
        for site in range(1, L + 1):
            ln = site - 1 if which % 2 == 0 else L - site
            cnt, buf = C.c_int32(), np.zeros(1 << 16, np.uint8)
            assert lib.tci_batch_indexset(b, i, which, site, C.byref(cnt), tci._abi.u8ptr(buf), len(buf)) == 0
            out.append(buf[:cnt.value * ln].reshape(cnt.value, ln).tolist())
    return out


@pytest.mark.parametrize("order", ["first", "last", "accessors"])
def test_accessors_agree(tci, ctx, order):
    sp = specs()
    b = _submit(tci, ctx, [_tci_problem(tci, s) for s in sp])
    lib = tci._abi.lib()
    try:
        idx = list(range(len(sp)))
        for i in idx[::-1] if order == "last" else idx:
            L = len(sp[i][4])
            if order == "accessors":
                direct = _sets(tci, b, i, L)
            t = tci.TensorCI2(b, i, sp[i][4])
            _check(t, sp[i])
            if order != "accessors":
                direct = _sets(tci, b, i, L)
            hist = (t.Iset_history + t.Jset_history) or [[[] for _ in range(L)]] * 2
            assert t.Iset + t.Jset + hist[0] + hist[1] == direct
            for site, x in enumerate(t.sitetensors):
                d3, out = np.zeros(3, np.int64), np.zeros(x.size)
                assert lib.tci_batch_sitetensor(b, i, site + 1, tci._abi.i64ptr(d3), tci._abi.dptr(out), out.size) == 0
                assert tuple(d3) == x.shape and np.array_equal(out, x.ravel(order="F"))
    finally:
        assert lib.tci_batch_free(b) == 0


def test_failed_solves_among_others(tci, ctx):
    ok = (tci.Lorentz(1.0), [10] * 5, None, dict(tolerance=1e-8))
    zero = (tci.Lorentz(0.0), [2] * 5, None, {})
    small = (tci.Lorentz(1.0), [10] * 8, None, dict(tolerance=1e-12, chi_cap=4, maxiter=3))
    ts = tci.crossinterpolate2_batch([zero, ok, small, ok, zero])
    assert [t.status for t in ts] == [4, 0, 10, 0, 4]
    assert ts[0].sitetensors == [] and ts[2].sitetensors == []
    assert ts[1].Iset == ts[3].Iset and all(np.array_equal(x, y) for x, y in zip(ts[1].sitetensors, ts[3].sitetensors))
    (alone,) = tci.crossinterpolate2_batch([ok])
    assert alone.Iset == ts[1].Iset and alone.Jset_history == ts[1].Jset_history
