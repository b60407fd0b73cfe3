"""TT evaluation over points grouped by local index, against the oracle's chain
bit for bit (abstracttensortrain.jl:124-132), where its tiles can go wrong:
groups of one point, of exactly 64 and of one more, local dimensions up to the
largest, bonds at the edges of a wave's columns and of the unrolled products,
and both sides of the rule that picks the route."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _train(rng, ds, chis):
    k = [1] + list(chis) + [1]
    return [rng.standard_normal((k[b], ds[b], k[b + 1])) / np.sqrt(k[b]) for b in range(len(ds))]


@pytest.mark.parametrize("ds,chis,npts", [
    ([3, 2, 4, 2], [9, 33, 8], 3000),          # odd bonds, remainders of every kind
    ([1, 5, 1, 3, 1], [17, 16, 15, 31], 1500),  # sites with one index: one group
    ([2] * 6, [32, 64, 65, 63, 32], 128),       # groups of about 64
    ([255, 254, 3], [40, 41], 700),             # more groups than tiles' worth of points
    ([4, 6, 4], [256, 255], 300),               # the widest bonds it takes
    ([4, 6, 4], [257, 40], 300),                # beyond them: the other route
    ([7, 3, 5], [12, 13], 1),                   # one point: the other route
    ([6, 3, 5, 8], [60, 61, 62], 97),           # just enough work
])
def test_grouped_equals_oracle(tci, ctx, ds, chis, npts):
    rng = np.random.default_rng(sum(chis) + npts)
    cores = _train(rng, ds, chis)
    x = np.stack([rng.integers(1, d + 1, npts) for d in ds], 1).astype(np.uint8)
    print("grouped", ds, chis, npts, flush=True)
    assert np.array_equal(tci.tt_evaluate(cores, x), O.tt_evaluate(cores, x.astype(np.int32)))


@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_group_sizes_around_a_tile(tci, ctx, extra):
    rng = np.random.default_rng(5)
    ds, chis = [3, 3, 3], [90, 90]
    cores = _train(rng, ds, chis)
    n = 64 + extra
    x = np.concatenate([np.full((n, 3), 1), np.full((1, 3), 2), np.full((2 * n, 3), 3)]).astype(np.uint8)
    x = x[rng.permutation(len(x))]
    assert np.array_equal(tci.tt_evaluate(cores, x), O.tt_evaluate(cores, x.astype(np.int32)))


def test_nan_and_infinite_cores(tci, ctx):
    rng = np.random.default_rng(6)
    cores = _train(rng, [3, 4, 3], [40, 50])
    cores[1][3, 1, 7], cores[1][5, 2, 9] = np.nan, np.inf
    x = np.stack([rng.integers(1, d + 1, 900) for d in (3, 4, 3)], 1).astype(np.uint8)
    assert np.array_equal(tci.tt_evaluate(cores, x), O.tt_evaluate(cores, x.astype(np.int32)), equal_nan=True)
