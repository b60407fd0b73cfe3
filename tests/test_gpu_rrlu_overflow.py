"""Entries whose squares overflow in the on-chip rrLU kernel whose members keep
columns outside the registers (tci_rrlu_chip.hip): all such entries tie, so the first
position wins (matrixlu.jl:1-32), whatever column of a member holds them and however far
apart their values are."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

GRID = 3
S, CB = 256, 4    # members of the team and register columns of each, 4097 to 8192 rows and more


# columns of one member, all outside its registers: both in LDS, LDS and memory, both
# in memory; the rows 512 apart, so that one thread holds both entries
@pytest.mark.parametrize("e1,e2", [(0, 1), (1, 3), (2, 4)])
@pytest.mark.parametrize("values", [(1e160, 2e160), (3e155, -1e300), (-1e200, np.inf)])
def test_overflowed_squares_tie(tci, ctx, e1, e2, values):
    m, n, g = 6400, S * (CB + 5), 77
    rng = np.random.default_rng(e1 + 10 * e2)
    A = np.asfortranarray(rng.standard_normal((m, 3)) @ rng.standard_normal((3, n)))
    c1, c2 = g + S * (CB + e1), g + S * (CB + e2)
    A[200, c1], A[200 + 512, c2] = values
    print("overflow", m, n, e1, e2, values, flush=True)
    c = tci.Context(0)
    try:
        assert tci._abi.lib().tci_ctx_set_rrlu_algo(c.handle, GRID) == 0
        for lo in (True, False):
            try:
                b, code = O.rrlu(A, maxrank=3, leftorthogonal=lo), 0
            except O.OracleError as e:
                b, code = None, e.code
            if code:
                with pytest.raises(tci.TCIError) as err:
                    tci.rrlu(A, ctx=c, maxrank=3, leftorthogonal=lo)
                assert err.value.status == code
                continue
            a = tci.rrlu(A, ctx=c, maxrank=3, leftorthogonal=lo)
            assert (b.rowpermutation[0], b.colpermutation[0]) == (201, c1 + 1)
            assert a.npivot == b.npivot and a.error == b.error
            assert np.array_equal(a.rowpermutation, b.rowpermutation)
            assert np.array_equal(a.colpermutation, b.colpermutation)
            assert np.array_equal(a.L, b.L) and np.array_equal(a.U, b.U)
    finally:
        c.close()
