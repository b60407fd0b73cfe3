"""Host staging of large batches: batch after batch its memory is used again instead of
being unmapped and mapped anew (page faults counted), and what an earlier batch left in
it reaches no later one's results."""
import ctypes as C
import resource

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _run(tci, c, f, dims, n):
    lib = tci._abi.lib()
    h = tci._holder(f, dims, None, dict(tolerance=1e-8))
    arr = (tci._abi.tci_problem * n)(*[h.st] * n)
    b = C.c_void_p()
    tci._check(lib.tci_solve_submit(c.handle, n, arr, C.byref(b)))
    try:
        tci._check(lib.tci_batch_wait(b))
        return tci.TensorCI2(b, n - 1, dims)
    finally:
        tci._check(lib.tci_batch_free(b))


def test_staging_is_used_again(tci, ctx):
    c = tci.Context(0)
    try:
        for _ in range(4):
            _run(tci, c, tci.Lorentz(1.0), [10] * 8, 4096)
        before = resource.getrusage(resource.RUSAGE_SELF).ru_minflt
        for _ in range(4):
            _run(tci, c, tci.Lorentz(1.0), [10] * 8, 4096)
        faults = (resource.getrusage(resource.RUSAGE_SELF).ru_minflt - before) / 4
        print("page faults a batch:", faults, flush=True)
        assert faults < 1000   # 6 MB each of inputs and reports are 3000 pages
        # smaller and differently shaped batches behind large ones
        for kind, dims, n in ((1.0, [10] * 8, 3000), (2.0, [4] * 6, 1500), (0.5, [3, 7, 2, 9, 5], 2500)):
            t = _run(tci, c, tci.Lorentz(kind), dims, n)
            o, ranks, errors = O.crossinterpolate2(O.Functor(1, [kind]), dims, tolerance=1e-8)
            assert t.status == 0 and list(t.ranks) == list(ranks) and np.array_equal(t.errors, errors)
            for b in range(len(dims)):
                assert t.Iset[b] == o.Iset(b) and np.array_equal(t.sitetensors[b], o.sitetensor(b))
    finally:
        c.close()
