"""Column pairs whose overlap lies at the convergence threshold to within the rounding of a dot
product: two Gram matrices summed in different orders disagree about them, and the iteration ends
all the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("block", [32, 16])
@pytest.mark.parametrize("m,n", [(2048, 256), (1000, 320)])
def test_overlaps_at_the_threshold(ctx, m, n, block):
    import direct_svd
    print(f"borderline svd {m}x{n} block {block}", flush=True)
    rng = np.random.default_rng(m + n + block)
    q, _ = np.linalg.qr(rng.standard_normal((m, n)))
    # lengths fall from column to column, so that the iteration keeps their order
    length = 1.0 - 1e-3 * np.arange(n)
    a = q * length
    norm = np.linalg.norm(length)
    # one pair of columns for each pair of column blocks
    nb = n // block
    eps = np.linspace(-2e-4, 2e-4, nb * (nb - 1) // 2)
    rng.shuffle(eps)
    pairs = [(i * block + j % block, j * block + i % block) for i in range(nb)
             for j in range(i + 1, nb)]
    for (x, y), e in zip(pairs, eps):
        lx, ly = length[x], length[y]
        thr = max(1e-13 * lx * ly, 1e-14 * norm * (lx + ly))
        a[:, y] += q[:, x] * (thr / lx * (1.0 + e))
    # not preconditioned: the columns are rotated as they are
    ((w, v, s),), sweeps, worst = direct_svd.decompose(ctx, [a], precondition=0, block=block)
    # the flagged pairs rotate in the first sweep; a second and third may find some again
    assert worst == 0.0 and sweeps <= 5
    np.testing.assert_allclose(s, np.sort(np.linalg.svd(a, compute_uv=False)), rtol=1e-12)
    np.testing.assert_allclose(v.T @ v, np.eye(n), rtol=0, atol=1e-12)
    np.testing.assert_allclose(w, a @ v, rtol=0, atol=1e-12)
