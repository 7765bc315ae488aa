"""SVDs of small and large LDS blocks at the same time, one context per thread: the kernel's LDS
limit is the function's, so no thread may set it to its own batch's need just before another's
launch.  Every result equals the one a thread gets alone, bit for bit."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_contexts_on_threads():
    from su2dmrg_amd import lib as L
    rng = np.random.default_rng(0)
    mats = [rng.standard_normal(s) for s in ((4, 3), (96, 96), (20, 31), (128, 70))]

    def call(ctx, a):
        m, n = a.shape
        # a sector of zeros keeps none of its columns, so a cut is possible
        t = L.wavefunction(ctx, [1, 3], [m, 3], [n, 2], {1: a})
        U, V, kept, _ = L.svd_truncate(ctx, t, 1.0, 0.0, min(m, n) + 1)
        return U[1], V[1], np.array(kept)

    ctxs = [L.Context(0) for _ in mats]
    alone = [call(c, a) for c, a in zip(ctxs, mats)]
    bad = []

    def work(i):
        try:
            for _ in range(100):
                got = call(ctxs[i], mats[i])
                if not all(np.array_equal(x, y) for x, y in zip(got, alone[i])):
                    bad.append(i)
        except Exception as e:   # noqa: BLE001 (reported by the assertion below)
            bad.append(e)

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(mats))]
    for x in th:
        x.start()
    for x in th:
        x.join()
    for c in ctxs:
        c.close()
    assert not bad
