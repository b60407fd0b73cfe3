"""The floating-zone search (globalsearch.jl:43-95) on the device against the
oracle, bit for bit, where its kernel can go wrong: functors of per-site terms
and others, one site, more indices per site than a wave has lanes, bonds at the
edges of eight loads, trains whose slices, then whose work area, do not fit in
LDS, and more starts than workgroups."""
import numpy as np
import pytest

import oracle as O
from problems import GSUM, LORENTZ, WLORENTZ, gauss_sum, random_tt

pytestmark = pytest.mark.gpu


def _functor(kind, L, d):
    if kind == WLORENTZ:
        return np.concatenate([[float(d)], np.linspace(0.5, 2.0, L)])
    return gauss_sum(3, L, max(d, 2), L) if kind == GSUM else [1.0]


@pytest.mark.parametrize("kind", [WLORENTZ, GSUM, LORENTZ])
@pytest.mark.parametrize("bonds,ld,n", [
    ([1, 1], [5], 3), ([1, 8, 1], [64, 65], 20), ([1, 7, 9, 1], [3, 200, 2], 40),
    ([1, 16, 17, 16, 1], [4] * 4, 300), ([1, 40, 40, 40, 1], [6] * 4, 30), ([1, 130, 130, 1], [30, 30, 30], 12),
    ([1, 4, 4, 1], [3, 3, 3], 2100)])
def test_floatingzone_edges(tci, ctx, kind, bonds, ld, n):
    L = len(ld)
    print("zone", kind, bonds, ld, n, flush=True)
    cores = random_tt(bonds, ld, sum(bonds) + n)[2]
    par = _functor(kind, L, max(ld))
    of = O.Functor(kind, par, [])
    df = tci.DeviceFunctor(kind, np.asarray(par, float), np.zeros(0, np.int32))
    rng = np.random.default_rng(n)
    starts = np.stack([rng.integers(1, d + 1, n) for d in ld], 1)
    for kw in (dict(), dict(nsweeps=2, earlystoptol=1e6)):
        piv, errs = tci.floatingzone(tci.TensorTrain(cores), df, starts, ctx=ctx, **kw)
        opiv, oerrs = O.floatingzone(of, cores, starts, **kw)
        assert np.array_equal(piv, opiv) and np.array_equal(errs, oerrs)


def test_floatingzone_nan_and_equal_errors(tci, ctx):
    # equal errors keep the first index; NaN errors are above all, the first of them wins
    tab = np.ones((70, 3))
    tab[66, 1] = tab[40, 1] = np.nan
    tab[3, 2] = np.inf
    of, df = O.Functor(6, tab.ravel(order="F"), [70, 3]), tci.TableFunctor(tab)
    cores = [np.zeros((1, 70, 1)), np.ones((1, 3, 1))]
    starts = np.array([[1, 1], [70, 2], [67, 3], [5, 3]])
    piv, errs = tci.floatingzone(tci.TensorTrain(cores), df, starts, ctx=ctx)
    opiv, oerrs = O.floatingzone(of, cores, starts)
    assert np.array_equal(piv, opiv) and np.array_equal(errs, oerrs, equal_nan=True)
