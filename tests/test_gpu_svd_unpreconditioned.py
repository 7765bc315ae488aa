"""Preconditioning switched off, or on from a limit only: the block Jacobi iteration on the columns
as they are, for blocks of every size past one compute unit's LDS."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


# (rows, columns, rank, decades): the sizes are outside the LDS kernel's
@pytest.mark.parametrize("limit", [0, 512])
@pytest.mark.parametrize("m,n,rank,decades", [(97, 97, 97, 6), (300, 20, 20, 8), (150, 129, 100, 12),
                                              (200, 255, 200, 10), (300, 257, 257, 6)])
def test_off_below_the_limit(ctx, m, n, rank, decades, limit):
    from su2dmrg_amd import lib as L
    print(f"unpreconditioned svd {m}x{n} rank {rank} limit {limit}", flush=True)
    rng = np.random.default_rng(m + 5 * n)
    k = min(m, n)
    u, _ = np.linalg.qr(rng.standard_normal((m, rank)))
    v, _ = np.linalg.qr(rng.standard_normal((n, rank)))
    a = (u * np.logspace(0, -decades, rank)) @ v.T
    t = L.wavefunction(ctx, [1, 3], [m, 3], [n, 2], {1: a})
    out = {}
    for lim in (256, limit):
        ctx.set_svd_precondition(lim)
        # the sector of zeros keeps none of its two columns: a cut is possible
        out[lim] = L.svd_truncate(ctx, t, 0.0, 1.0, k + 1)
    ctx.set_svd_precondition(256)
    # the reflectors change the last bits
    assert not np.array_equal(out[limit][0][1], out[256][0][1])
    ref = np.sort(np.linalg.svd(a, compute_uv=False))
    for U, V, kept, _ in out.values():
        s = np.array(kept)
        # the bounds of the other block tests: values to 1e-12 of the largest, the product to
        # 1e-13 and the weight of the columns zeroed at s <= 1e-11 s_max, U's columns orthogonal
        # to 1e-13 s_max / s where s > 1e-9 s_max
        np.testing.assert_allclose(s, ref[k - s.size:], rtol=0, atol=1e-12 * ref[-1])
        cut = s[s <= 1e-11 * s[-1]].sum()
        np.testing.assert_allclose(U[1] @ V[1].T, a, rtol=0, atol=1e-13 * ref[-1] + cut)
        big = s > 1e-9 * s[-1]
        ub, sb = U[1][:, big], s[big]
        bound = 1e-13 * s[-1] / np.minimum.outer(sb, sb) + 1e-13
        assert np.all(np.abs(ub.T @ ub - np.eye(big.sum())) <= bound)
