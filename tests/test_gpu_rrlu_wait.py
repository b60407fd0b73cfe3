"""Teams of the on-chip rrLU (tci_rrlu_chip.hip) that give up a wait: with no time to
wait at all, every job of a launch reports either TCI_ERR_DEVICE or its right result,
those that no workgroup had begun included, and the kernel ends as it always does."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

ERR_DEVICE = 12


def _lowrank(rng, m, n, r):
    return rng.standard_normal((m, r)) @ rng.standard_normal((r, n)) + 1e-12 * rng.standard_normal((m, n))


# teams of 4 (more of them than fit the device at once), lone members among them; and
# teams of the kernel with columns in LDS
@pytest.mark.parametrize("shapes,count", [([(300, 250), (140, 20), (300, 250)], 900), ([(3080, 2600)], 3)])
def test_waits_given_up(tci, ctx, monkeypatch, shapes, count):
    rng = np.random.default_rng(count)
    some = [_lowrank(rng, m, n, 6) for m, n in shapes]
    want = [O.rrlu(A, reltol=1e-9) for A in some]
    mats = [some[q % len(some)] for q in range(count)]
    monkeypatch.setenv("TCI_RRLU_WAIT_MS", "0")
    hasty = tci.Context(0)
    monkeypatch.delenv("TCI_RRLU_WAIT_MS")
    patient = tci.Context(0)
    try:
        for c, failing in ((hasty, True), (patient, False)):
            print("wait given up", failing, shapes, count, flush=True)
            res = tci.rrlu_batched(mats, reltol=1e-9, ctx=c)
            bad = 0
            for q, r in enumerate(res):
                o = want[q % len(some)]
                if r["status"] == ERR_DEVICE:
                    assert r["npivot"] == 0 and shapes[q % len(some)][1] != 20
                    bad += 1
                    continue
                assert r["status"] == 0 and r["npivot"] == o.npivot and r["error"] == o.error, q
                assert np.array_equal(r["rowpermutation"], o.rowpermutation), q
                assert np.array_equal(r["colpermutation"], o.colpermutation), q
            assert (bad > 0) == failing
    finally:
        hasty.close()
        patient.close()
