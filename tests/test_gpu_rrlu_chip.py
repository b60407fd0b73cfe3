"""The on-chip rrLU kernels (tci_rrlu_chip.hip) against the oracle, bit for
bit, where they can go wrong: matrix sides at the edges of the register
shapes (rows of a wave, of all its wave rows; columns of one member and of
one more), the shapes whose columns spill to LDS and memory, ties, zeros,
subnormal squares, infinities and NaN, a maximum rank, and one launch over
many uneven matrices whose teams differ (matrixlu.jl:141-181)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

GRID, STREAM = 3, 1


@pytest.fixture
def chip_ctx(tci, ctx):
    c = tci.Context(0)
    assert tci._abi.lib().tci_ctx_set_rrlu_algo(c.handle, GRID) == 0
    yield c
    c.close()


def _lowrank(rng, m, n, r):
    return rng.standard_normal((m, r)) @ rng.standard_normal((r, n)) + 1e-12 * rng.standard_normal((m, n))


def _check(tci, ctx, A, **kw):
    print("chip case", A.shape, kw, flush=True)
    try:
        b, st = O.rrlu(A, **kw), 0
    except O.OracleError as e:
        b, st = None, e.code
    try:
        a, ast = tci.rrlu(A, ctx=ctx, **kw), 0
    except tci.TCIError as e:
        a, ast = None, e.status
    assert ast == st
    if st:
        return
    assert a.npivot == b.npivot
    assert np.array_equal(a.rowpermutation, b.rowpermutation)
    assert np.array_equal(a.colpermutation, b.colpermutation)
    assert a.error == b.error or (np.isnan(a.error) and np.isnan(b.error))
    assert np.array_equal(a.L, b.L) and np.array_equal(a.U, b.U)


# rows at the edges of 64·WR·RA; columns at the edges of one member's share
@pytest.mark.parametrize("m", [64, 65, 128, 129, 192, 193, 256, 257, 320, 321, 384, 385, 512, 513, 769, 1025, 1281])
def test_row_edges(tci, chip_ctx, m):
    rng = np.random.default_rng(m)
    for n, lo in ((22, True), (169, False)):
        _check(tci, chip_ctx, _lowrank(rng, m, n, 9), reltol=1e-10, leftorthogonal=lo)


@pytest.mark.parametrize("n", [1, 2, 41, 42, 43, 87, 88, 89, 168, 169, 337])
def test_column_edges(tci, chip_ctx, n):
    rng = np.random.default_rng(n)
    for m, lo in ((100, False), (250, True), (1000, True)):
        _check(tci, chip_ctx, _lowrank(rng, m, n, min(7, n)), reltol=1e-10, leftorthogonal=lo)


# the kernel whose members keep columns in LDS and memory: each of its shapes,
# with columns in registers only, in LDS too, and in memory too
@pytest.mark.parametrize("m,n", [(3071, 2900), (3073, 2600), (3200, 3900), (4609, 1300), (4700, 2700), (6145, 1100),
                                 (8192, 1500)])
def test_big_shapes(tci, chip_ctx, m, n):
    rng = np.random.default_rng(m + n)
    A = np.asfortranarray(_lowrank(rng, m, n, 12))
    _check(tci, chip_ctx, A, reltol=1e-10, leftorthogonal=m % 2 == 0)


@pytest.mark.parametrize("m,n", [(90, 70), (300, 250), (700, 900), (3100, 2700)])
def test_special_values(tci, chip_ctx, m, n):
    rng = np.random.default_rng(m)
    mr = 24
    ties = rng.integers(-2, 3, (m, n)).astype(float)
    for lo in (True, False):
        _check(tci, chip_ctx, ties, maxrank=mr, leftorthogonal=lo)
    _check(tci, chip_ctx, np.zeros((m, n)), maxrank=mr)
    _check(tci, chip_ctx, -np.zeros((m, n)), maxrank=mr)
    _check(tci, chip_ctx, _lowrank(rng, m, n, 5) * 1e-160, maxrank=mr)   # subnormal squares
    _check(tci, chip_ctx, _lowrank(rng, m, n, 5) * 1e-200, maxrank=mr)   # squares of 0
    one = _lowrank(rng, m, n, 5)
    for value in (np.inf, np.nan):
        A = one.copy()
        A[m // 2, n // 3] = value
        for lo in (True, False):
            _check(tci, chip_ctx, A, maxrank=mr, leftorthogonal=lo)
    _check(tci, chip_ctx, np.full((m, n), np.nan), maxrank=mr)
    _check(tci, chip_ctx, one, maxrank=1)
    _check(tci, chip_ctx, one, abstol=1e-3)


@pytest.mark.parametrize("seed", range(3))
def test_many_uneven_matrices_in_one_launch(tci, ctx, seed):
    """Packed factors and permutations equal the streaming kernel's, pivots
    and errors the oracle's; more teams than fit the device at once."""
    import torch
    rng = np.random.default_rng(seed)
    mats = []
    for q in range(160):
        m, n = (int(v) for v in rng.integers(1, 700 if q % 8 else 1500, 2))
        mats.append(_lowrank(rng, m, n, int(rng.integers(1, 1 + min(m, n, 20)))))
    dev, offs, shapes = tci.upload_matrices(mats)
    got, outs = [], []
    for algo in (0, STREAM):
        c = tci.Context(0)
        assert tci._abi.lib().tci_ctx_set_rrlu_algo(c.handle, algo) == 0
        A = dev.clone()
        got.append(tci.rrlu_batched(None, reltol=1e-9, leftorthogonal=seed != 1, ctx=c, device_buffers=(A, offs, shapes)))
        outs.append(A)
        c.close()
    assert torch.equal(outs[0], outs[1])
    for q, (a, b) in enumerate(zip(*got)):
        assert a["npivot"] == b["npivot"] and a["status"] == b["status"] == 0 and a["error"] == b["error"], q
        assert np.array_equal(a["rowpermutation"], b["rowpermutation"]), q
        assert np.array_equal(a["colpermutation"], b["colpermutation"]), q
    for q in range(0, 160, 16):
        o = O.rrlu(mats[q], reltol=1e-9, leftorthogonal=seed != 1)
        assert got[0][q]["npivot"] == o.npivot and got[0][q]["error"] == o.error
