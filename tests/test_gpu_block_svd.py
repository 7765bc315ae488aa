"""Sector blocks past one CU's LDS, with a possible cut, against LAPACK.

Such calls take the preconditioned block Jacobi (an uncut call keeps the plain iteration, which
test_gpu_dmrg covers): pairs of 32-column blocks rotated against each other, whole blocks in their
first visit of a sweep, only the pairs that still need it.  Sizes just past the LDS limit, a last
column block of one column, a block far taller than wide, and rank-deficient ones; both column block widths and up to three inner sweeps.
"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("block,inner", [(32, 1), (32, 3), (16, 1)])
@pytest.mark.parametrize("m,n,rank,decades", [
    (97, 97, 97, 6), (300, 20, 20, 8), (129, 129, 129, 12), (200, 193, 130, 12),
    (255, 400, 255, 3), (260, 257, 150, 14), (700, 560, 400, 13)])
def test_block_against_lapack(ctx, m, n, rank, decades, block, inner):
    # the bounds of test_gpu_dmrg's plain runs: values to 1e-12 of the largest, the product to
    # 1e-13 and the weight of the columns zeroed at s <= 1e-11 s_max, the short side orthonormal
    # to 1e-11
    from su2dmrg_amd import lib as L
    print(f"block svd {m}x{n} rank {rank}, block {block}, inner {inner}", flush=True)
    sys.stdout.flush()
    ctx.set_svd_tuning(block, inner)
    rng = np.random.default_rng(m + 3 * n)
    k = min(m, n)
    u, _ = np.linalg.qr(rng.standard_normal((m, k)))
    v, _ = np.linalg.qr(rng.standard_normal((n, k)))
    s = np.zeros(k)
    s[:rank] = np.logspace(0, -decades, rank)
    a = (u * s) @ v.T
    # a sector of zeros keeps no column, so the limit below cuts none, but might
    t = L.wavefunction(ctx, [1, 3], [m, 3], [n, 2], {1: a})
    p1, p2 = (1.0, 0.0) if m >= n else (0.0, 1.0)
    U, V, kept, _ = L.svd_truncate(ctx, t, p1, p2, k + 1)
    ctx.set_svd_tuning(32, 1)
    ref = np.sort(np.linalg.svd(a, compute_uv=False))
    got = np.array(kept)
    np.testing.assert_allclose(got, ref[k - got.size:], rtol=0, atol=1e-12 * ref[-1])
    cut = got[got <= 1e-11 * got[-1]].sum()
    np.testing.assert_allclose(U[1] @ V[1].T, a, rtol=0, atol=1e-13 * ref[-1] + cut)
    q = V[1] if m >= n else U[1]
    np.testing.assert_allclose(q.T @ q, np.eye(q.shape[1]), rtol=0, atol=1e-11)
