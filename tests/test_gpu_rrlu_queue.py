"""The asynchronous batched rrLU followed by the calls that use the same host tables
(one matrix, MatrixLUCI, compress!, another batch) with nothing waited for in between:
every result equals the oracle's."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _lowrank(rng, m, n, r):
    return rng.standard_normal((m, r)) @ rng.standard_normal((r, n)) + 1e-12 * rng.standard_normal((m, n))


def _batch(tci, mats):
    import torch
    A, offs, shapes = tci.upload_matrices(mats)
    perm = torch.zeros(sum(m + n for m, n in shapes), dtype=torch.int32, device=A.device)
    jobs = (tci._abi.tci_lu_job * len(mats))()
    o = 0
    for j, off, (m, n) in zip(jobs, offs, shapes):
        j.A = A.data_ptr() + 8 * off
        j.rowperm = perm.data_ptr() + 4 * o
        j.colperm = perm.data_ptr() + 4 * (o + m)
        j.m, j.n, j.maxrank, j.reltol, j.leftorth = m, n, tci.TCI_UNLIMITED, 1e-9, 1
        o += m + n
    jb = torch.frombuffer(bytearray(jobs), dtype=torch.uint8).to(A.device)
    torch.cuda.synchronize()
    return A, perm, jb, jobs


def test_calls_behind_a_queued_batch(tci, ctx, monkeypatch):
    monkeypatch.setenv("TCI_TT_FUSED", "0")   # compress! bond by bond, through the rrLU kernels
    rng = np.random.default_rng(5)
    big = [_lowrank(rng, 700 + 3 * q, 650 - 2 * q, 60) for q in range(48)]
    mixed = [_lowrank(rng, int(m), int(n), 5) for m, n in rng.integers(20, 400, (60, 2))]
    links = [1, 6, 20, 40, 20, 6, 1]
    cores = [rng.standard_normal((links[b], 6, links[b + 1])) for b in range(6)]
    one, two = _lowrank(rng, 330, 310, 20), _lowrank(rng, 90, 100, 12)
    tt = tci.TensorTrain(cores)
    c = tci.Context(0)
    try:
        batches = [_batch(tci, big), _batch(tci, mixed), _batch(tci, big)]

        def queue(b):
            print("queued batch of", len(b[3]), flush=True)
            assert tci._abi.lib().tci_rrlu_batched_f64(c.handle, C.c_void_p(b[2].data_ptr()), len(b[3])) == 0

        queue(batches[0])
        first = tci.rrlu(one, reltol=1e-9, ctx=c)
        queue(batches[1])
        tci.compress(tt, "LU", tolerance=1e-8, ctx=c)
        queue(batches[2])
        last = tci.rrlu(two, reltol=1e-9, ctx=c)
        luci = tci.MatrixLUCI(one, reltol=1e-9, ctx=c)
        c.synchronize()
    finally:
        c.close()
    for A, got in ((one, first), (two, last)):
        o = O.rrlu(A, reltol=1e-9)
        assert got.npivot == o.npivot and got.error == o.error
        assert np.array_equal(got.rowpermutation, o.rowpermutation) and np.array_equal(got.L, o.L)
        assert np.array_equal(got.colpermutation, o.colpermutation) and np.array_equal(got.U, o.U)
    assert list(luci.rowindices()) == list(O.rrlu(one, reltol=1e-9).rowpermutation[:first.npivot])
    for x, y in zip(tt.sitetensors, O.tt_compress(cores, "LU", tolerance=1e-8)):
        assert np.array_equal(x, y)
    for (A, perm, jb, jobs), mats in zip(batches, (big, mixed, big)):
        C.memmove(jobs, jb.cpu().numpy().tobytes(), C.sizeof(jobs))
        permh, at = perm.cpu().numpy(), 0
        for j, M in zip(jobs, mats):
            o = O.rrlu(M, reltol=1e-9)
            assert j.status == 0 and j.npivot == o.npivot and j.error == o.error
            assert np.array_equal(permh[at:at + M.shape[0]], o.rowpermutation)
            assert np.array_equal(permh[at + M.shape[0]:at + sum(M.shape)], o.colpermutation)
            at += sum(M.shape)
