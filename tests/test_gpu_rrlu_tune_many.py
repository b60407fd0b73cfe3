"""A tuned context and a batch of more jobs than the autotuner times in one launch
(tci_ctx_set_rrlu_tuning, grid_max_jobs 64): the batch stays on the on-chip kernel, also
beside jobs whose entry allows none.  Results against the oracle, routes by time, in
between those of a table without on-chip jobs and of the fixed rules."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _table(*rows):
    return [dict(side=s, tile=0, grid_team=256, grid_max_jobs=k) for s, k in rows]


@pytest.mark.parametrize("small,rows", [(0, [(8192, 64)]), (40, [(192, 0), (8192, 64)])])
def test_large_batch_on_a_tuned_context(tci, ctx, small, rows):
    import torch
    rng = np.random.default_rng(small)
    mats = [rng.standard_normal((512, 64)) @ rng.standard_normal((64, 480)) for _ in range(4)] * 40
    mats += [rng.standard_normal((150, 8)) @ rng.standard_normal((8, 140))] * small
    dev, offs, shapes = tci.upload_matrices(mats)
    c = tci.Context(0)
    ms = {}
    try:
        for name, table in (("fixed", []), ("tuned", _table(*rows)), ("streamed", _table((8192, 0)))):
            c.set_rrlu_tuning(table)
            times = []
            for _ in range(4):
                A = dev.clone()
                e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
                torch.cuda.synchronize()
                e[0].record()
                res = tci.rrlu_batched(None, reltol=1e-9, ctx=c, device_buffers=(A, offs, shapes))
                e[1].record()
                torch.cuda.synchronize()
                times.append(e[0].elapsed_time(e[1]))
            ms[name] = min(times)
            for q in (0, 1, len(mats) - 1):
                o = O.rrlu(mats[q], reltol=1e-9)
                assert res[q]["status"] == 0 and res[q]["npivot"] == o.npivot and res[q]["error"] == o.error
                assert np.array_equal(res[q]["colpermutation"], o.colpermutation)
    finally:
        c.close()
    print("tuned large batch, ms:", ms, flush=True)
    assert ms["tuned"] < 0.5 * (ms["fixed"] + ms["streamed"])
