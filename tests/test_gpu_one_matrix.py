"""One factorization at a time (tci_rrlu_f64, tci_luci_f64) and the kernels
behind the tensor-train sweeps, at the edges of their dispatch: LUCI factors
at ranks around the unrolled step of the substitution, around the largest
rank it takes, and with the smaller side beyond that rank; strides larger
than the matrix; matrices that go up in one piece or two, and results that
come down in one piece or two; products at the edges of a tile, with signed
zeros, infinities and NaN; sweeps around the fused sweep's largest bond
matrix.  All bit for bit."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from problems import random_tt

pytestmark = pytest.mark.gpu


def _one(tci, ctx, fn, A, lda, ldx, ldy, maxrank, reltol, lo):
    """The entry point with its own strides; what lies between columns is kept."""
    m, n = A.shape
    store = np.full((lda, n), -7.0, order="F")
    store[:m] = A
    cap = min(m, n, maxrank)
    X = np.full((ldx, cap), -7.0, order="F")
    Y = np.full((ldy, n), -7.0, order="F")
    rp, cp = np.zeros(m, np.int64), np.zeros(n, np.int64)
    p, err = C.c_int64(), C.c_double()
    ab = tci._abi
    print(fn, A.shape, lda, ldx, ldy, maxrank, lo, flush=True)
    tci._check(getattr(ab.lib(), fn)(ctx.handle, ab.dptr(store), lda, m, n, maxrank, reltol, 0.0, int(lo),
                                     ab.i64ptr(rp), ab.i64ptr(cp), ab.dptr(X), ldx, ab.dptr(Y), ldy,
                                     C.byref(p), C.byref(err)))
    p = p.value
    assert np.all(X[m:] == -7.0) and np.all(X[:, p:] == -7.0) and np.all(Y[p:] == -7.0)
    assert np.all(store[m:] == -7.0) and np.array_equal(store[:m], A)
    return p, rp, cp, X[:m, :p], Y[:p], err.value


def _both(tci, ctx, A, pad=(0, 0, 0), maxrank=1 << 30, reltol=1e-12, lo=True):
    m, n = A.shape
    cap = min(m, n, maxrank)
    kw = dict(maxrank=maxrank, reltol=reltol, leftorthogonal=lo)
    lu, left, right = O.luci_factors(A, **kw)
    for fn, X, Y in (("tci_rrlu_f64", lu.L, lu.U), ("tci_luci_f64", left, right)):
        p, rp, cp, x, y, err = _one(tci, ctx, fn, A, m + pad[0], m + pad[1], cap + pad[2], maxrank, reltol, lo)
        assert p == lu.npivot and err == lu.error
        assert np.array_equal(rp, lu.rowpermutation) and np.array_equal(cp, lu.colpermutation)
        assert np.array_equal(x, X) and np.array_equal(y, Y)


@pytest.mark.parametrize("lo", [True, False])
@pytest.mark.parametrize("rank", [1, 7, 8, 9, 17, 64])
def test_ranks(tci, ctx, rank, lo):
    rng = np.random.default_rng(rank)
    A = rng.standard_normal((71, 65))
    _both(tci, ctx, A, maxrank=rank, lo=lo)
    _both(tci, ctx, A.T.copy(order="F"), pad=(3, 1, 2), maxrank=rank, lo=lo)


@pytest.mark.parametrize("lo", [True, False])
@pytest.mark.parametrize("m,n,rank", [(260, 300, 255), (300, 260, 256), (260, 300, 257), (300, 270, 40),
                                      (1, 5, 1), (5, 1, 1), (64, 64, 64), (128, 1024, 20), (363, 362, 10)])
def test_sides_and_stages(tci, ctx, m, n, rank, lo):
    # 128×1024 doubles are the largest that go up in one piece; 363×362 go up by columns
    A = np.random.default_rng(m + n).standard_normal((m, n))
    _both(tci, ctx, A, maxrank=rank, lo=lo)
    _both(tci, ctx, A, pad=(2, 5, 1), maxrank=rank, lo=lo)


def test_large_results(tci, ctx):
    # (1100 + 1090)·500 doubles are more than 8 MB: L and U come down after the
    # rank, in one piece at rank 30, column by column at rank 500
    rng = np.random.default_rng(8)
    for A in (rng.standard_normal((1100, 30)) @ rng.standard_normal((30, 1090)), rng.standard_normal((1100, 1090))):
        _both(tci, ctx, A, maxrank=500, reltol=1e-10)
        _both(tci, ctx, A, pad=(1, 3, 2), maxrank=500, reltol=1e-10, lo=False)


@pytest.mark.parametrize("M,N,K", [(32, 32, 16), (33, 31, 17), (31, 65, 15), (64, 1, 33), (1, 33, 1), (5, 5, 0)])
def test_product(tci, ctx, M, N, K):
    rng = np.random.default_rng(M * N + K)
    A = np.asfortranarray(rng.standard_normal((M, K)))
    B = np.asfortranarray(rng.standard_normal((K, N)))
    if K > 1:
        A[0, 0], A[M // 2, K - 1], B[K // 2, 0], B[0, N // 2] = np.inf, -0.0, np.nan, -np.inf
    out = np.full((M, N), -7.0, order="F")
    ab = tci._abi
    tci._check(ab.lib().tci_gemm_f64(ctx.handle, M, N, K, ab.dptr(A) if A.size else None, M,
                                     ab.dptr(B) if B.size else None, max(K, 1), ab.dptr(out), M))
    ref = np.zeros((M, N))
    with np.errstate(invalid="ignore"):
        for k in range(K):
            ref = ref + np.multiply.outer(A[:, k], B[k, :])
    assert np.array_equal(out, ref, equal_nan=True)
    num = ~np.isnan(ref)
    assert np.array_equal(np.signbit(out[num]), np.signbit(ref[num]))


# bond matrices just under, at and above the fused sweep's limits, in the mean and the largest
@pytest.mark.parametrize("chi,d", [(32, 2), (32, 3), (33, 3), (55, 1), (47, 2), (48, 2), (56, 2)])
@pytest.mark.parametrize("method", ["LU", "CI"])
def test_sweep_limit(tci, ctx, chi, d, method):
    cores = random_tt([1, chi, chi, chi, 1], [d] * 4, chi + d)[2]
    tt = tci.TensorTrain(cores)
    tci.compress(tt, method, tolerance=1e-10, ctx=ctx)
    ref = O.tt_compress(cores, method, tolerance=1e-10)
    assert len(ref) == len(tt.sitetensors)
    for x, y in zip(tt.sitetensors, ref):
        assert np.array_equal(x, y)
