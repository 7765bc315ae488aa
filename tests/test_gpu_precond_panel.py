"""Preconditioned SVD of blocks whose columns come in nearly parallel groups, so that reflectors of
one panel start from columns that almost depend on those before them; sizes around the panel width
(a last panel of one column, a full one, a block of two panels)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("spread", [1e-2, 1e-6, 1e-9, 0.0])
@pytest.mark.parametrize("m,n,group", [(97, 97, 2), (130, 112, 16), (113, 150, 5), (300, 257, 40)])
def test_nearly_parallel_columns(ctx, m, n, group, spread):
    # the bounds of the other block tests: values to 1e-12 of the largest, the product to 1e-13
    # and the weight of the columns zeroed at s <= 1e-11 s_max, the short side orthonormal to 1e-11
    from su2dmrg_amd import lib as L
    print(f"svd {m}x{n}, groups of {group} columns {spread} apart", flush=True)
    rng = np.random.default_rng(m + n + group)
    k, big = min(m, n), max(m, n)
    lead = rng.standard_normal((big, (k + group - 1) // group))
    a = np.repeat(lead, group, axis=1)[:, :k] + spread * rng.standard_normal((big, k))
    if m < n:
        a = a.T
    t = L.wavefunction(ctx, [1, 3], [m, 3], [n, 2], {1: a})
    p1, p2 = (1.0, 0.0) if m >= n else (0.0, 1.0)
    U, V, kept, _ = L.svd_truncate(ctx, t, p1, p2, k + 1)
    ref = np.sort(np.linalg.svd(a, compute_uv=False))
    got = np.array(kept)
    np.testing.assert_allclose(got, ref[k - got.size:], rtol=0, atol=1e-12 * ref[-1])
    cut = got[got <= 1e-11 * got[-1]].sum()
    np.testing.assert_allclose(U[1] @ V[1].T, a, rtol=0, atol=1e-13 * ref[-1] + cut)
    q = V[1] if m >= n else U[1]
    np.testing.assert_allclose(q.T @ q, np.eye(q.shape[1]), rtol=0, atol=1e-11)
