"""Factorizations beyond the solve team's register tile: extended tiles, whose
columns beyond the registers lie in LDS and in memory, against the oracle bit
for bit, at the edges of their shapes and areas.  On the CPU the tile code runs
on 256 host threads shaped like four waves; on the GPU whole solves have bond
matrices of these sizes."""
import ctypes as C

import numpy as np
import pytest

import eh
import oracle as O
from problems import GSUM, WLORENTZ, gauss_sum

SHAPES = [(4, 18), (3, 24), (2, 32), (4, 4)]   # doubles per lane: rows, columns


def _ext(shape, n1, n2, inplace, A, maxrank, reltol, lo):
    m, n = A.shape
    W = np.array(A, order="F")
    rp, cp = np.zeros(m, np.int32), np.zeros(n, np.int32)
    L = np.zeros((m, n), order="F")
    err = C.c_double()
    d, i = C.POINTER(C.c_double), C.POINTER(C.c_int32)
    f = eh.lib().eh_rrlu_ext_mt
    f.argtypes = [C.c_int, C.c_int64, C.c_int64, C.c_int, d, C.c_int, C.c_int, C.c_int64, C.c_double, C.c_double,
                  C.c_int, i, i, d, d]
    p = f(shape, n1, n2, inplace, W.ctypes.data_as(d), m, n, maxrank, reltol, 0.0, int(lo), rp.ctypes.data_as(i),
          cp.ctypes.data_as(i), L.ctypes.data_as(d), C.byref(err))
    return p, rp + 1, cp + 1, L, err.value


def _cases(shape, area):
    ra, cb = SHAPES[shape]
    mr, reg = 64 * ra, 4 * cb   # rows and register columns of four waves
    sizes = ((mr, reg), (mr - 1, 255), (65, reg + 9)) if area == "two" else ((mr, reg + 1), (mr - 63, 256), (1, 200))
    for m, n in sizes:
        yield m, min(n, 256)


@pytest.mark.parametrize("shape", range(4))
@pytest.mark.parametrize("area", ["one", "two", "memory", "inplace"])
def test_ext_tile_equals_oracle(shape, area):
    rng = np.random.default_rng(10 * shape + len(area))
    for t, (m, n) in enumerate(_cases(shape, area)):
        per = 4 * m   # doubles of one more column per wave
        n1, n2 = {"one": (64 * per, 0), "two": (3 * per + 1, 2 * per), "memory": (0, per - 1), "inplace": (0, 0)}[area]
        if t % 3 == 0:
            A = rng.standard_normal((m, 7)) @ rng.standard_normal((7, n)) + 1e-12 * rng.standard_normal((m, n))
        elif t % 3 == 1:
            A = rng.integers(-1, 2, (m, n)).astype(float)     # ties and zeros
        else:
            A = rng.standard_normal((m, n))
            A[rng.random((m, n)) < 0.02] = np.nan
        for lo, rank in ((t % 2 == 0, 8),):
            try:
                b, st = O.rrlu(A, maxrank=rank, reltol=1e-10, leftorthogonal=lo), 0
            except O.OracleError as e:
                b, st = None, e.code
            p, rp, cp, L, err = _ext(shape, n1, n2, area == "inplace", A, rank, 1e-10, lo)
            if st:
                assert p == -st
                continue
            assert p == b.npivot and err == b.error
            assert np.array_equal(rp, b.rowpermutation) and np.array_equal(cp, b.colpermutation)
            for k in range(p):   # columns of L, by original row
                assert np.array_equal(L[rp[k + 1:] - 1, k], b.L[k + 1:, k])


def test_ext_tile_tiny_magnitudes():
    """Squares that are subnormal or zero: the first of many equal ones."""
    rng = np.random.default_rng(5)
    for scale in (1e-158, 1e-162):
        A = rng.standard_normal((130, 90)) * scale
        b = O.rrlu(A, maxrank=4, reltol=0.0)
        p, rp, cp, L, err = _ext(0, 1000, 20000, 0, A, 4, 0.0, True)
        assert p == b.npivot and err == b.error
        assert np.array_equal(rp, b.rowpermutation) and np.array_equal(cp, b.colpermutation)


# bond matrices of d·χ rows and columns: just beyond the team's tile, at the ends of
# the row shapes (192, 256) and beyond them; wide, narrow, and of a rook search
@pytest.mark.gpu
@pytest.mark.parametrize("ld,opts", [
    ([130, 130], dict(maxbonddim=40)), ([192, 255], dict(maxbonddim=30)), ([193, 255], dict(maxbonddim=20)),
    ([255, 33], dict(maxbonddim=30)), ([200, 32], dict(maxbonddim=30)), ([64, 250], dict(maxbonddim=30)),
    ([128, 129], dict(maxbonddim=30)), ([16] * 6, dict(maxbonddim=14)), ([64] * 4, dict(maxbonddim=4)),
    ([43] * 4, dict(maxbonddim=6)), ([48] * 4, dict(maxbonddim=6, pivotsearch="rook")),
    ([16] * 6, dict(maxbonddim=256)), ([13] * 5, dict(maxbonddim=256, normalizeerror=False))])
def test_solves_beyond_the_tile(tci, ctx, ld, opts):
    from test_gpu_solves import _check, _tci_problem
    n = len(ld)
    rng = np.random.default_rng(sum(ld) + n)
    opts = dict(tolerance=1e-9, maxiter=4, **opts)
    for kind, par in ((GSUM, gauss_sum(3, n, max(ld), n)),
                      (WLORENTZ, np.concatenate([[float(max(ld))], rng.uniform(0.5, 2, n)]))):
        print("solve", kind, ld, opts, flush=True)
        spec = ("ext", kind, par, [], ld, None, opts)
        (t,) = tci.crossinterpolate2_batch([_tci_problem(tci, spec)])
        _check(t, spec)
