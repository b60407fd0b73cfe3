"""Performance cases of the TCI framework: what its users run, through the
public entry points of the package, over the ranges they run it on.

A case is a dict of plain values; `kind` picks the path:

  lorentz     crossinterpolate2 of a / (1 + v.v) (the README example)
  quantics    crossinterpolate2 of a sum of Gaussians and a cosine on 2^L points
  highdim     crossinterpolate2 of 1 / (1 + sum c_i (v_i/16)^2) in many dimensions
  mix         a batch of uneven Gaussian-sum problems, as a server meets them
  rrlu        rank-revealing LU of one host matrix
  rrlu_batch  rank-revealing LU of matrices resident on the device
  tt_eval     a tensor train evaluated at many points
  compress    a redundant tensor train recompressed
  to_tci2     a tensor train converted to a TensorCI2
  true_error  the search for the largest |f - TT| of a finished interpolation

Every solve of a batch has parameters of its own.  Outputs are the whole
result of the call: index sets, errors and site tensors of a solve, packed
factors and permutations of a factorization, cores of a train.
"""
import importlib.util
import math
import os
import sys
from itertools import chain

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _pkg():
    if "tci_amd" in sys.modules:
        return sys.modules["tci_amd"]
    pkg = os.path.join(ROOT, "tensorcrossinterpolation.jl_amd")
    spec = importlib.util.spec_from_file_location("tci_amd", os.path.join(pkg, "__init__.py"),
                                                  submodule_search_locations=[pkg])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["tci_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


tci = _pkg()


def listed():
    return [
        # one interactive call: a single small interpolation, latency is all that counts
        dict(name="lorentz_one", kind="lorentz", L=8, d=10, tol=1e-8, count=1),
        # a parameter scan of the same function: throughput of many small solves
        dict(name="lorentz_batch", kind="lorentz", L=8, d=10, tol=1e-8, count=384),
        # quantics: long chains of d = 2 with an expensive function
        dict(name="quantics_batch", kind="quantics", L=30, K=6, tol=1e-10, maxbond=200, count=48),
        # many dimensions with a large local dimension: Pi matrices of a few hundred rows
        dict(name="highdim", kind="highdim", L=40, d=16, tol=1e-10, maxbond=256, count=3),
        # what a service holds at one moment: uneven problems of 4 to 12 sites, d from 2 to 32
        dict(name="served_mix", kind="mix", tol_lo=1e-10, tol_hi=1e-6, maxbond=128, count=96),
        # one small odd-sized matrix on the host: the smallest call there is
        dict(name="rrlu_small", kind="rrlu", m=97, n=83, rank=31, reltol=1e-10, leftorth=True),
        # a batch of uneven matrices resident on the device
        dict(name="rrlu_batch", kind="rrlu_batch", count=1024, lo=32, hi=1024, rank_lo=8, rank_hi=128,
             maxrank=1 << 40, reltol=1e-10, leftorth=True),
        # one bond of an L = 40, d = 16 interpolation at bond dimension 256
        dict(name="rrlu_bond", kind="rrlu_batch", count=1, lo=4352, hi=4352, rank_lo=300, rank_hi=300,
             maxrank=256, reltol=1e-14, leftorth=True),
        # a finished train sampled for plots or checks
        dict(name="tt_eval", kind="tt_eval", L=20, d=10, chi=96, npts=100000),
        # the sum of a few trains brought back to its true rank
        dict(name="compress", kind="compress", L=20, d=16, chi=128, rank=80, tol=1e-8, method="LU"),
        # a train from elsewhere (a solver, a sum) turned into an interpolation
        dict(name="to_tci2", kind="to_tci2", L=16, d=12, chi=72, rank=50, tol=1e-12),
        # the error estimate after a solve, from random starts
        dict(name="true_error", kind="true_error", L=20, d=16, tol=1e-7, npts=2000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lorentz", "quantics", "highdim", "mix", "rrlu", "rrlu_batch", "rrlu_batch", "tt_eval",
                       "compress", "to_tci2", "true_error"])
    if kind == "lorentz":
        return dict(kind=kind, L=rng.randint(4, 8), d=rng.randint(3, 10), tol=10.0 ** rng.uniform(-9, -5),
                    count=_log(rng, 1, 384))
    if kind == "quantics":
        return dict(kind=kind, L=rng.randint(10, 30), K=rng.randint(1, 6), tol=10.0 ** rng.uniform(-10, -6),
                    maxbond=200, count=_log(rng, 1, 48))
    if kind == "highdim":
        return dict(kind=kind, L=rng.randint(6, 40), d=rng.randint(3, 16), tol=10.0 ** rng.uniform(-10, -6),
                    maxbond=256, count=rng.randint(1, 3))
    if kind == "mix":
        return dict(kind=kind, tol_lo=1e-10, tol_hi=1e-6, maxbond=128, count=_log(rng, 4, 96))
    if kind == "rrlu":
        m, n = _log(rng, 8, 700), _log(rng, 8, 700)
        return dict(kind=kind, m=m, n=n, rank=rng.randint(1, min(m, n)), reltol=1e-10, leftorth=rng.random() < 0.5)
    if kind == "rrlu_batch":
        if rng.random() < 0.5:   # a few large matrices
            lo = _log(rng, 256, 4000)
            hi = rng.randint(lo, min(4352, lo + lo // 4))
            return dict(kind=kind, count=rng.randint(1, 4), lo=lo, hi=hi, rank_lo=lo // 16, rank_hi=lo // 8,
                        maxrank=256, reltol=1e-12, leftorth=rng.random() < 0.5)
        hi = _log(rng, 48, 1024)
        lo = rng.randint(16, hi)
        rank_lo = max(1, min(64, lo // 4))
        return dict(kind=kind, count=_log(rng, 2, 768), lo=lo, hi=hi, rank_lo=rank_lo,
                    rank_hi=max(rank_lo, min(128, hi // 4)), maxrank=1 << 40, reltol=1e-10,
                    leftorth=rng.random() < 0.5)
    if kind == "tt_eval":
        return dict(kind=kind, L=rng.randint(3, 30), d=rng.randint(2, 16), chi=_log(rng, 2, 96),
                    npts=_log(rng, 10, 60000))
    if kind == "compress":
        chi = _log(rng, 4, 128)
        return dict(kind=kind, L=rng.randint(4, 20), d=rng.randint(2, 16), chi=chi, rank=rng.randint(1, chi),
                    tol=10.0 ** rng.uniform(-10, -6), method=rng.choice(["LU", "CI"]))
    if kind == "to_tci2":
        chi = _log(rng, 3, 72)
        return dict(kind=kind, L=rng.randint(4, 16), d=rng.randint(2, 12), chi=chi, rank=rng.randint(1, chi),
                    tol=10.0 ** rng.uniform(-12, -8))
    return dict(kind=kind, L=rng.randint(5, 20), d=rng.randint(2, 16), tol=10.0 ** rng.uniform(-8, -5),
                npts=_log(rng, 20, 2000))


# ------------------------------------------------------------------- inputs
def _mix_shapes(count):
    """(K, sites, d) of each problem of a mix: the same mix for every seed."""
    rng = np.random.default_rng([count, 18])
    return [(int(rng.integers(1, 9)), int(rng.integers(4, 13)), int(rng.choice([2, 4, 8, 16, 32])))
            for _ in range(count)]


def _dims(case):
    """The local dimensions of every problem of a solve case."""
    if case["kind"] == "mix":
        return [[d] * n for _, n, d in _mix_shapes(case["count"])]
    return [[case.get("d", 2)] * case["L"]] * case["count"]


def _problems(case, seed):
    """The problems of one solve case: (functor, localdims, initial pivots, keywords)."""
    rng = np.random.default_rng([seed, 11])
    shapes = _mix_shapes(case["count"])
    kind, out = case["kind"], []
    for q, dims in enumerate(_dims(case)):
        if kind == "lorentz":
            f = tci.Lorentz(rng.uniform(0.5, 2.0))
            kw = dict(tolerance=case["tol"])
        elif kind == "quantics":
            K = case["K"]
            f = tci.QuanticsGaussCos(rng.uniform(0.5, 2, K), rng.uniform(0, 1, K), 10.0 ** rng.uniform(-6, -1, K),
                                     0.1, 2.0 ** 20)
            kw = dict(tolerance=case["tol"], maxbonddim=case["maxbond"])
        elif kind == "highdim":
            f = tci.WeightedLorentz(rng.uniform(0.5, 2, case["L"]))
            kw = dict(tolerance=case["tol"], maxbonddim=case["maxbond"])
        else:
            K, n, d = shapes[q]
            f = tci.GaussSum(rng.uniform(0.5, 2, K), rng.uniform(0.2, 0.6, K), rng.uniform(0, 1, (K, n)), d)
            kw = dict(tolerance=float(10.0 ** rng.uniform(np.log10(case["tol_lo"]), np.log10(case["tol_hi"]))),
                      maxbonddim=case["maxbond"])
        out.append((f, dims, None, kw))
    return out


def _host_matrix(case, seed):
    rng = np.random.default_rng([seed, 12])
    m, n, r = case["m"], case["n"], case["rank"]
    return np.asfortranarray(rng.standard_normal((m, r)) @ rng.standard_normal((r, n))
                             + 1e-12 * rng.standard_normal((m, n)))


def _device_matrices(case, seed):
    """Matrices X·Y + 1e-12·E, column-major back to back on the device; the
    shapes are those of the case, the same for every seed."""
    rng = np.random.default_rng([case["count"], case["lo"], case["hi"], 13])
    c = case["count"]
    ms, ns = rng.integers(case["lo"], case["hi"] + 1, c), rng.integers(case["lo"], case["hi"] + 1, c)
    rs = rng.integers(case["rank_lo"], case["rank_hi"] + 1, c)
    offs = np.concatenate([[0], np.cumsum(ms * ns)])
    A = torch.empty(int(offs[-1]), dtype=torch.float64, device="cuda")
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    for m, n, r, o in zip(ms.tolist(), ns.tolist(), rs.tolist(), offs.tolist()):
        X = torch.randn(m, r, dtype=torch.float64, device="cuda", generator=g)
        Y = torch.randn(r, n, dtype=torch.float64, device="cuda", generator=g)
        # (the transpose, row-major, is the matrix in column-major order)
        T = torch.randn(n, m, dtype=torch.float64, device="cuda", generator=g).mul_(1e-12)
        A[o:o + m * n] = T.addmm_(Y.t().contiguous(), X.t().contiguous()).view(-1)
    return A, [int(o) for o in offs[:-1]], [(int(m), int(n)) for m, n in zip(ms, ns)]


def _links(L, d, chi):
    return [min(chi, d ** min(b, L - b, 30)) for b in range(L + 1)]


def _random_train(L, d, chi, rng):
    k = _links(L, d, chi)
    return [rng.standard_normal((k[b], d, k[b + 1])) / math.sqrt(k[b] * d) for b in range(L)]


def _redundant_train(case, seed):
    """A train of true rank `rank` carried with bond dimension `chi`: at each
    bond Q·Q⁺ = 1 is inserted, Q of `chi` columns, with a little noise."""
    rng = np.random.default_rng([seed, 14])
    cores = _random_train(case["L"], case["d"], case["rank"], rng)
    for b in range(case["L"] - 1):
        r = cores[b].shape[2]
        q = rng.standard_normal((r, max(r, case["chi"])))
        cores[b] = np.tensordot(cores[b], q, 1)
        cores[b] += 1e-12 * rng.standard_normal(cores[b].shape) * np.abs(cores[b]).max()
        cores[b + 1] = np.tensordot(np.linalg.pinv(q), cores[b + 1], 1)
    return [np.asfortranarray(c) for c in cores]


def _points(L, d, npts, seed):
    return np.random.default_rng([seed, 15]).integers(1, d + 1, (npts, L)).astype(np.uint8)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("lorentz", "quantics", "highdim", "mix"):
        s["problems"] = _problems(case, seed)
    elif kind == "rrlu":
        s["A"] = _host_matrix(case, seed)
    elif kind == "rrlu_batch":
        s["A"], s["offs"], s["shapes"] = _device_matrices(case, seed)
    elif kind == "tt_eval":
        s["cores"] = _random_train(case["L"], case["d"], case["chi"], np.random.default_rng([seed, 16]))
        s["points"] = _points(case["L"], case["d"], case["npts"], seed)
    elif kind in ("compress", "to_tci2"):
        s["cores"] = _redundant_train(case, seed)
    elif kind == "true_error":
        # the train of a finished interpolation, and the points to start from
        rng = np.random.default_rng([seed, 17])
        s["f"] = tci.WeightedLorentz(rng.uniform(0.5, 2, case["L"]))
        t, _, _ = tci.crossinterpolate2(float, s["f"], [case["d"]] * case["L"], tolerance=case["tol"], maxbonddim=64)
        s["tt"] = tci.TensorTrain(t)
        s["points"] = _points(case["L"], case["d"], case["npts"], seed)
    else:
        raise ValueError(kind)
    return s


# --------------------------------------------------------------------- runs
def _fill(parts, total, dtype=np.float64):
    """The parts back to back in an array of `total` values, zeros after
    them: ranks differ from input to input, the size of the output does not."""
    flat = np.concatenate([np.zeros(0, dtype), *parts])
    if len(flat) > total:
        raise ValueError("%d values, room for %d" % (len(flat), total))
    out = np.zeros(total, dtype)
    out[:len(flat)] = flat
    return out


def _ints(nested, total):
    """Lists of multi-indices as one array."""
    return _fill([np.fromiter(chain.from_iterable(chain.from_iterable(nested)), np.int64)], total, np.int64)


def _flat(cores, total):
    return _fill([c.ravel(order="F") for c in cores], total)


def _elems(cores):
    return sum(c.size for c in cores)


def _room(dims, chi):
    """Values of the site tensors and of the index sets of a train."""
    k = [_links(len(d), d[0], chi) for d in dims]
    return (sum(q[b] * d[b] * q[b + 1] for q, d in zip(k, dims) for b in range(len(d))),
            sum(q[b] * b for q, d in zip(k, dims) for b in range(len(d))))


# no solve of the declared ranges ends with a larger bond dimension
MOST_CHI = {"lorentz": 16, "quantics": 40, "highdim": 24, "mix": 24}
MAXITER = 20


def _solutions(ts, case):
    """The whole result of a batch of solves."""
    count, chi = case["count"], MOST_CHI[case["kind"]]
    tensors, sets = _room(_dims(case), chi)
    history = np.zeros((3, count, MAXITER))
    for i, t in enumerate(ts):
        for row, v in zip(history, (t.ranks, t.errors, t.nglobalpivots)):
            row[i, :len(v)] = v
    return dict(
        status=np.array([t.status for t in ts]),
        linkdims=np.concatenate([t.linkdims() for t in ts]),
        history=history,
        maxsample=np.array([t.maxsamplevalue for t in ts]),
        pivoterrors=_fill([t.pivoterrors for t in ts], count * (chi + 1)),
        bonderrors=np.concatenate([t.bonderrors for t in ts]),
        Iset=_ints((s for t in ts for s in t.Iset), sets),
        Jset=_ints((s for t in ts for s in t.Jset), sets),
        sitetensors=_flat([x for t in ts for x in t.sitetensors], tensors),
    )


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("lorentz", "quantics", "highdim", "mix"):
        return _solutions(tci.crossinterpolate2_batch(state["problems"]), case)
    if kind == "rrlu":
        lu = tci.rrlu(state["A"], reltol=case["reltol"], leftorthogonal=case["leftorth"])
        return dict(rows=lu.rowpermutation, cols=lu.colpermutation, L=lu.L, U=lu.U, npivot=lu.npivot, error=lu.error)
    if kind == "rrlu_batch":
        # the factorization overwrites its input: the program keeps its matrices
        A = state["A"].clone()
        res = tci.rrlu_batched(None, maxrank=case["maxrank"], reltol=case["reltol"],
                               leftorthogonal=case["leftorth"], device_buffers=(A, state["offs"], state["shapes"]))
        return dict(A=A, rows=np.concatenate([r["rowpermutation"] for r in res]),
                    cols=np.concatenate([r["colpermutation"] for r in res]),
                    npivot=np.array([r["npivot"] for r in res]), error=np.array([r["error"] for r in res]),
                    status=np.array([r["status"] for r in res]))
    if kind == "tt_eval":
        return tci.tt_evaluate(state["cores"], state["points"])
    if kind == "compress":
        tt = tci.TensorTrain(state["cores"])
        tci.compress(tt, case["method"], tolerance=case["tol"])
        return dict(linkdims=np.array(tt.linkdims()), cores=_flat(tt.sitetensors, _elems(state["cores"])))
    if kind == "to_tci2":
        t = tci.tensorci2_from_tt(tci.TensorTrain(state["cores"]), tolerance=case["tol"])
        sets = case["L"] ** 2 * case["chi"]
        return dict(linkdims=np.array(t.linkdims()), Iset=_ints(t.Iset, sets), Jset=_ints(t.Jset, sets),
                    pivoterrors=t.pivoterrors, maxsample=t.maxsamplevalue,
                    sitetensors=_flat(t.sitetensors, _elems(state["cores"])))
    found = tci.estimatetrueerror(state["tt"], state["f"], initialpoints=state["points"])
    return dict(pivots=_ints([[p for p, _ in found]], case["npts"] * case["L"]),
                errors=_fill([np.array([e for _, e in found])], case["npts"]))


# --------------------------------------------------------------------- work
def _lu_work(m, n, p, top):
    """Bytes and flops of rrlu of an m×n matrix with p pivots: the matrix read
    and its packed factors written once; two flops per Schur update."""
    p = min(p, m, n, top)
    k = np.arange(1, p + 1, dtype=np.float64)
    return 16.0 * m * n, float(2 * np.sum((m - k) * (n - k)))


def _train_elems(L, d, chi):
    k = _links(L, d, chi)
    return float(sum(k[b] * d * k[b + 1] for b in range(L)))


def work(case):
    """What a pass cannot do without.  The rank of a solve is not known
    beforehand: the figures use the rank the function class ends with, one
    factorization per bond and half-sweep, four iterations of two half-sweeps."""
    kind = case["kind"]
    if kind in ("lorentz", "quantics", "highdim", "mix"):
        if kind == "mix":
            L, d, chi, per = 8, 12, 14, 200.0
        else:
            L, d = case["L"], case.get("d", 2)
            chi = {"lorentz": 12, "quantics": 18, "highdim": 14}[kind]
            per = {"lorentz": 2.0 * L, "quantics": 60.0 * case.get("K", 0), "highdim": 4.0 * L}[kind]
        side = chi * d
        nlu = 8.0 * (L - 1)
        flops = nlu * (2.0 * side * side * chi + per * side * side)
        return {"bytes": case["count"] * 8.0 * _train_elems(L, d, chi), "flops": case["count"] * flops}
    if kind == "rrlu":
        b, f = _lu_work(case["m"], case["n"], case["rank"], case["m"])
        return {"bytes": b, "flops": f}
    if kind == "rrlu_batch":
        side, rank = 0.5 * (case["lo"] + case["hi"]), 0.5 * (case["rank_lo"] + case["rank_hi"])
        b, f = _lu_work(int(side), int(side), int(rank), case["maxrank"])
        return {"bytes": case["count"] * b, "flops": case["count"] * f}
    if kind == "tt_eval":
        e = _train_elems(case["L"], case["d"], case["chi"])
        return {"bytes": 8.0 * e + case["npts"] * (case["L"] + 8.0), "flops": 2.0 * case["npts"] * e / case["d"]}
    if kind in ("compress", "to_tci2"):
        k = _links(case["L"], case["d"], case["chi"])
        flops = 0.0
        for b in range(1, case["L"]):
            m, n, p = k[b - 1] * case["d"], k[b], min(k[b], case["rank"])
            flops += 2 * (_lu_work(m, n, p, m)[1] + 2.0 * n * n * case["d"] * k[b + 1])
        return {"bytes": 16.0 * _train_elems(case["L"], case["d"], case["chi"]), "flops": flops}
    e = _train_elems(case["L"], case["d"], 12)
    return {"bytes": 8.0 * e + 2.0 * case["npts"] * case["L"],
            "flops": 3.0 * case["npts"] * (2.0 * e + 4.0 * case["L"] * case["L"] * case["d"])}


# -------------------------------------------------------------------- exact
def _numpy_rrlu(A, reltol, leftorth):
    """Full-pivoting rank-revealing LU of a small matrix, one pivot at a time."""
    A = np.array(A, order="F")
    m, n = A.shape
    rows, cols = np.arange(m), np.arange(n)
    err, top, p = math.nan, 0.0, 0
    for k in range(min(m, n)):
        j, i = divmod(int(np.argmax(np.square(A[k:, k:]).ravel(order="F"))), m - k)
        i, j = i + k, j + k
        err = abs(A[i, j])
        if k > 0 and err < reltol * top:
            break
        top = max(top, err)
        A[[k, i]], rows[[k, i]] = A[[i, k]], rows[[i, k]]
        A[:, [k, j]], cols[[k, j]] = A[:, [j, k]], cols[[j, k]]
        if leftorth:
            A[k + 1:, k] /= A[k, k]
        else:
            A[k, k + 1:] /= A[k, k]
        A[k + 1:, k + 1:] -= np.outer(A[k + 1:, k], A[k, k + 1:])
        p = k + 1
    if p >= min(m, n):
        err = 0.0
    L, U = np.tril(A[:, :p]), np.triu(A[:p])
    np.fill_diagonal(L if leftorth else U, 1.0)
    return dict(rows=rows + 1, cols=cols + 1, L=L, U=U, npivot=p, error=err)


def exact(case, seed):
    kind = case["kind"]
    if kind == "rrlu":
        return _numpy_rrlu(_host_matrix(case, seed), case["reltol"], case["leftorth"])
    if kind == "tt_eval":
        s = prepare(case, seed)
        x = torch.from_numpy(s["points"].astype(np.int64) - 1)
        v = torch.ones(case["npts"], 1, dtype=torch.float64)
        for b, c in enumerate(s["cores"]):
            t = torch.from_numpy(np.ascontiguousarray(c.transpose(1, 0, 2)))
            w = torch.empty(case["npts"], t.shape[2], dtype=torch.float64)
            for q in range(case["d"]):
                at = torch.nonzero(x[:, b] == q).ravel()
                w[at] = v[at] @ t[q]
            v = w
        return v[:, 0].numpy()
    # pivots are chosen among nearly equal values along the way: a solve, a
    # large factorization or a sweep has no value that does not depend on
    # the order of its own roundings, or takes too long to restate
    return None
