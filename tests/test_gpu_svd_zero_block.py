"""Blocks of exact zeros: singular values of zero, an orthonormal V, and W of zeros, whatever kernel
the block's size sends it to."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("m,n", [(1, 1), (6, 5), (5, 6), (64, 64), (96, 96), (128, 70), (97, 97),
                                 (120, 300), (260, 257)])
def test_zero_block(ctx, m, n):
    import direct_svd
    print(f"zero block {m}x{n}", flush=True)
    (w, v, s), = direct_svd.decompose(ctx, [np.zeros((m, n))])[0]
    assert np.all(s == 0) and np.all(w == 0)
    # V is a product of reflectors with unit columns: k eps of its columns
    k = min(m, n)
    np.testing.assert_allclose(v.T @ v, np.eye(k), rtol=0, atol=1e-15 * k + 1e-15)
