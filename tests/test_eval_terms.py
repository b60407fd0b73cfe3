"""The solve engine's factored evaluations of f (per-site term tables of the
weighted Lorentzian and of Gaussian sums, split quantics coordinates) at the
edges of their rules: more sites to the right than a wave has lanes, the
most sites of a quantics function, tables beyond their size limit,
uneven local dimensions, parameters that give infinities, rows just past a
wave and a row block.  Every result equals the oracle bit for bit, on the
CPU build of the engine and on the device (batcheval.jl:32-61)."""
import numpy as np
import pytest

from problems import GSUM, QEXP, QGC, WLORENTZ, gauss_sum
from test_engine_host import _compare
from test_gpu_solves import _check, _tci_problem


def _cases():
    rng = np.random.default_rng(7)
    wl = lambda L: np.concatenate([[16.0], rng.uniform(0.5, 2, L)])   # noqa: E731
    few = dict(tolerance=1e-6, maxiter=4, maxbonddim=8)
    ragged = [3, 7, 2, 5, 33, 4]
    gs = gauss_sum(3, 6, 8, 4)
    inf = gauss_sum(2, 5, 1, 9)          # d - 1 = 0: infinite and NaN coordinates
    narrow = gauss_sum(2, 5, 6, 3)
    narrow[4:6] = 1e-3                   # exp underflows almost everywhere
    trip = np.array([1.0, 0.3, 0.2])
    return [
        ("terms_67_sites", WLORENTZ, wl(67), [], [2] * 67, None, dict(few, maxiter=2, nsearchglobalpivot=0)),
        ("terms_ragged", WLORENTZ, wl(6), [], ragged, None, few),
        ("terms_two_sites", WLORENTZ, wl(2), [], [65, 129], None, dict(tolerance=1e-8)),
        ("gauss_ragged", GSUM, gs, [], ragged, None, few),
        ("gauss_many", GSUM, gauss_sum(2300, 6, 10, 5), [], [10] * 6, None, dict(few, maxiter=1, maxbonddim=3)),
        ("gauss_underflow", GSUM, narrow, [], [6] * 5, [[3, 3, 3, 3, 3]], few),
        ("gauss_infinite", GSUM, inf, [], [1, 2, 2, 1, 2], None, dict(few, nsearchglobalpivot=0)),
        ("quantics_52", QGC, np.concatenate([[1], trip, [0.1, 64.0]]), [], [2] * 52, None, dict(few, maxiter=2)),
        ("quantics_digits", QEXP, [1.0, -1.0, 0.3, -2.0], [], [3, 2, 4, 2, 2, 5], None, few),
    ]


@pytest.mark.parametrize("spec", _cases(), ids=lambda s: s[0])
def test_host_engine(spec):
    _compare(spec, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 300])
def test_device(tci, ctx, count):
    """Alone (one solve per CU) and among many (two per CU)."""
    specs = _cases()
    ts = tci.crossinterpolate2_batch([_tci_problem(tci, s) for s in specs] * max(1, count // len(specs)))
    for q, t in enumerate(ts[:len(specs)] + ts[-len(specs):]):
        _check(t, specs[q % len(specs)])


@pytest.mark.gpu
@pytest.mark.parametrize("spec", _cases(), ids=lambda s: s[0])
def test_device_alone(tci, ctx, spec):
    print("solve", spec[0], flush=True)
    (t,) = tci.crossinterpolate2_batch([_tci_problem(tci, spec)])
    _check(t, spec)


