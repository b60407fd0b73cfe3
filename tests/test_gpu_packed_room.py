"""Reading results needs no device memory that the context's HBM budget does not have,
packs no more solves than a few for each one asked for, and gives the same values
whether a solve's results were packed or read piece by piece."""
import ctypes as C
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COUNT = 200


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _arr(tci, n):
    hs = [tci._holder(tci.Lorentz(1.0 + 1e-3 * (q % 7)), [10] * 8, None, dict(tolerance=1e-10)) for q in range(n)]
    return (tci._abi.tci_problem * n)(*[h.st for h in hs]), hs


def _same(a, b):
    assert a.Iset == b.Iset and a.Jset == b.Jset
    assert a.Iset_history == b.Iset_history and a.Jset_history == b.Jset_history
    assert len(a.sitetensors) == len(b.sitetensors) == 8
    assert all(np.array_equal(x, y) for x, y in zip(a.sitetensors, b.sitetensors))


def test_two_solves_of_many(tci, ctx):
    lib = tci._abi.lib()
    arr, keep = _arr(tci, COUNT)
    c, b = tci.Context(0), C.c_void_p()
    try:
        tci._check(lib.tci_solve_submit(c.handle, COUNT, arr, C.byref(b)))
        tci._check(lib.tci_batch_wait(b))
        before = _free()
        two = [tci.TensorCI2(b, i, [10] * 8) for i in (COUNT - 1, 3)]
        took = before - _free()
        rest = [tci.TensorCI2(b, i, [10] * 8) for i in range(COUNT)]
        all_bytes = sum(t.nbytes for r in rest for t in r.sitetensors)
        print("two solves took", took, "of", all_bytes, flush=True)
        assert took < all_bytes // 3
        _same(two[0], rest[COUNT - 1])
        _same(two[1], rest[3])
        for q in range(7, COUNT):
            _same(rest[q], rest[q % 7])
    finally:
        lib.tci_batch_free(b)
        c.close()


def test_budget_used_up(tci, ctx):
    lib = tci._abi.lib()
    arr, keep = _arr(tci, COUNT)
    b = C.c_void_p()
    tiny = tci.Context(0, 1 << 20)
    with pytest.raises(tci.TCIError) as e:
        tci._check(lib.tci_solve_submit(tiny.handle, COUNT, arr, C.byref(b)))
    tiny.close()
    need = int(re.search(r"batch needs (\d+) bytes", str(e.value)).group(1))
    want = tci.crossinterpolate2_batch([(tci.Lorentz(1.0 + 1e-3 * q), [10] * 8, None, dict(tolerance=1e-10))
                                        for q in range(7)])
    # nothing left, and room for a few solves' results
    for extra in (0, 1 << 20):
        c = tci.Context(0, need + extra)
        try:
            tci._check(lib.tci_solve_submit(c.handle, COUNT, arr, C.byref(b)))
            tci._check(lib.tci_batch_wait(b))
            before = _free()
            got = [tci.TensorCI2(b, i, [10] * 8) for i in range(COUNT)]
            took = before - _free()
            print("budget left", extra, "taken", took, flush=True)
            assert took <= max(2 * extra, 0)   # (allocations come in steps of 2 MiB)
            for q, t in enumerate(got):
                _same(t, want[q % 7])
            tci._check(lib.tci_batch_free(b))
            b = C.c_void_p()
            # the budget is whole again
            tci._check(lib.tci_solve_submit(c.handle, COUNT, arr, C.byref(b)))
        finally:
            lib.tci_batch_wait(b)
            lib.tci_batch_free(b)
            c.close()
