"""The SVD that the DMRG runs use (a cut is possible, so su2_svd_truncate takes the LDS kernel and
the preconditioned block Jacobi) under the bounds that test_gpu_dmrg.py puts on uncut calls: every
value to 1e-12 of the largest, the product to 1e-13 and the weight of the columns zeroed at
s <= 1e-11 s_max, the long side, which the rotations orthogonalise, to 1e-13 s_max / s, and the
uncut call's values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


def _block(m, n, decades, rank=None):
    rng = np.random.default_rng(m + n)
    k = rank or min(m, n)
    u, _ = np.linalg.qr(rng.standard_normal((m, k)))
    v, _ = np.linalg.qr(rng.standard_normal((n, k)))
    return (u * np.logspace(0, -decades, k)) @ v.T


def _svd(ctx, a, cut):
    """U, V, kept with the long side orthonormal and the short side carrying s."""
    from su2dmrg_amd import lib as L
    m, n = a.shape
    p1, p2 = (0.0, 1.0) if m >= n else (1.0, 0.0)
    if cut:   # a sector of zeros keeps none of its two columns
        t = L.wavefunction(ctx, [1, 3], [m, 3], [n, 2], {1: a})
        U, V, kept, _ = L.svd_truncate(ctx, t, p1, p2, min(m, n) + 1)
    else:
        t = L.wavefunction(ctx, [1], [m], [n], {1: a})
        U, V, kept, _ = L.svd_truncate(ctx, t, p1, p2, 100000)
    return U[1], V[1], np.array(kept)


def _check(a, res, ref, floor=1e-9, stop=False):
    U, V, s = res
    m, n = a.shape
    np.testing.assert_allclose(s, ref[ref.size - s.size:], rtol=0, atol=1e-12 * ref[-1])
    cut = s[s <= 1e-11 * s[-1]].sum()
    np.testing.assert_allclose(U @ V.T, a, rtol=0, atol=1e-13 * ref[-1] + cut)
    big = s > floor * s[-1]
    q, sb = (U if m >= n else V)[:, big], s[big]
    if stop:
        # where the iteration stops: |w_i.w_j| <= max(1e-13 |w_i||w_j|, 1e-14 |A| (|w_i| + |w_j|))
        bound = np.maximum(1e-13, 1e-14 * np.linalg.norm(s) * np.add.outer(1 / sb, 1 / sb)) + 1e-13
    else:
        bound = 1e-13 * s[-1] / np.minimum.outer(sb, sb) + 1e-13
    assert np.all(np.abs(q.T @ q - np.eye(big.sum())) <= bound)


@pytest.mark.parametrize("block,inner", [(32, 1), (32, 3), (16, 1)])
@pytest.mark.parametrize("m,n,decades", [(90, 80, 20), (64, 64, 12), (75, 120, 8), (96, 96, 16),
                                         (300, 200, 20), (180, 420, 12), (520, 500, 6),
                                         (700, 560, 14), (600, 1100, 8)])
def test_wide_spectrum(ctx, m, n, decades, block, inner):
    print(f"strict svd {m}x{n}, {decades} decades, block {block}, inner {inner}", flush=True)
    a = _block(m, n, decades)
    ctx.set_svd_tuning(block, inner)
    res = _svd(ctx, a, True)
    ctx.set_svd_tuning(32, 1)
    _check(a, res, np.sort(np.linalg.svd(a, compute_uv=False)))


@pytest.mark.parametrize("m,n,decades", [(90, 80, 10), (240, 200, 12), (700, 560, 14),
                                         (600, 1100, 8), (1300, 1290, 16)])
def test_both_iterations_and_preconditioning(ctx, m, n, decades):
    print(f"strict svd {m}x{n}, {decades} decades, all iterations", flush=True)
    a = _block(m, n, decades)
    ref = np.sort(np.linalg.svd(a, compute_uv=False))
    vals = []
    for cut in (True, False):
        for limit in (256, 48, 0):
            ctx.set_svd_precondition(limit)
            res = _svd(ctx, a, cut)
            _check(a, res, ref)
            vals.append(res[2])
    ctx.set_svd_precondition(256)
    for s in vals[1:]:
        k = min(s.size, vals[0].size)
        np.testing.assert_allclose(s[-k:], vals[0][-k:], rtol=0, atol=1e-12 * ref[-1])


@pytest.mark.parametrize("m,n,rank,gap", [(90, 96, 50, True), (92, 90, 60, False),
                                          (240, 200, 130, True), (200, 230, 150, False),
                                          (700, 720, 400, True), (530, 512, 300, False)])
def test_rank_deficient(ctx, m, n, rank, gap):
    # with a gap the nonzero values stop at 1e-10, without one they run down to 1e-14
    print(f"strict svd {m}x{n} of rank {rank}, gap {gap}", flush=True)
    a = _block(m, n, 10 if gap else 14, rank)
    ref = np.sort(np.linalg.svd(a, compute_uv=False))
    for limit in (256, 64, 0):
        ctx.set_svd_precondition(limit)
        res = _svd(ctx, a, True)
        # columns zeroed by convention are left out of the long side's test
        _check(a, res, ref, floor=1e-11)
        if gap:
            assert np.sum(res[2] > 1e-11 * res[2][-1]) == rank
    ctx.set_svd_precondition(256)


@pytest.mark.parametrize("m,n", [(2100, 2060), (2049, 2049)])
def test_past_the_preconditioner(ctx, m, n):
    # more than 2048 columns: rotated as they are
    print(f"strict svd {m}x{n}", flush=True)
    a = _block(m, n, 10)
    _check(a, _svd(ctx, a, True), np.sort(np.linalg.svd(a, compute_uv=False)), stop=True)
