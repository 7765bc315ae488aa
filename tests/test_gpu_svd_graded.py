"""Blocks whose columns (or rows) span many decades in no order, as the fused legs of a two-site
wavefunction have them: Jacobi's singular values are accurate relative to each value, not only to
the largest, on either side of the size that one compute unit takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("tall", [True, False])
@pytest.mark.parametrize("rows,cols", [(12, 9), (28, 24), (57, 48), (64, 64), (76, 64), (96, 90),
                                       (128, 70), (120, 110), (240, 200)])
def test_shuffled_column_grades(ctx, rows, cols, tall):
    import direct_svd
    print(f"graded svd {rows}x{cols} tall={tall}", flush=True)
    rng = np.random.default_rng(rows + cols)
    x = rng.standard_normal((rows, cols))
    d = np.logspace(0, -6, cols)
    a = x * rng.permutation(d)
    mat = a if tall else a.T
    (w, v, s), = direct_svd.decompose(ctx, [mat])[0]
    # values do not change with the order of the columns; bidiagonalised in descending order they
    # keep their relative accuracy
    order = np.argsort(-np.linalg.norm(a, axis=0))
    ref = np.linalg.svd(a[:, order], compute_uv=False)[::-1]
    # eps for each of the k rotations of a column, times the condition of the columns at unit
    # length (Demmel and Veselic)
    cond = np.linalg.cond(a / np.linalg.norm(a, axis=0))
    bound = cols * np.finfo(float).eps * cond
    assert np.max(np.abs(s - ref) / ref) < bound
    np.testing.assert_allclose(v.T @ v, np.eye(cols), rtol=0, atol=5e-13)
    work = mat if mat.shape[0] >= mat.shape[1] else mat.T
    np.testing.assert_allclose(w, work @ v, rtol=0, atol=5e-13)
