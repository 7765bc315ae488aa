"""A block so tall that a grouped GEMM cannot address the Gram matrix's operand (32-bit byte
offsets): decomposed all the same, with or without a possible cut."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("cut", [True, False])
def test_block_past_gemm_addressing(ctx, cut):
    from su2dmrg_amd import lib as L
    m, n = 2_000_000, 20
    print(f"tall svd {m}x{n}, cut possible: {cut}", flush=True)
    rng = np.random.default_rng(1)
    a = rng.standard_normal((m, n)) * np.logspace(0, -4, n)
    if cut:
        t = L.wavefunction(ctx, [1, 3], [m, 3], [n, 2], {1: a})
        U, V, kept, _ = L.svd_truncate(ctx, t, 0.0, 1.0, n + 1)
    else:
        t = L.wavefunction(ctx, [1], [m], [n], {1: a})
        U, V, kept, _ = L.svd_truncate(ctx, t, 0.0, 1.0, 100000)
    q, r = np.linalg.qr(a)
    ref = np.sort(np.linalg.svd(r, compute_uv=False))
    np.testing.assert_allclose(np.array(kept), ref, rtol=0, atol=1e-12 * ref[-1])
    np.testing.assert_allclose(U[1].T @ U[1], np.eye(n), rtol=0, atol=1e-11)
    np.testing.assert_allclose(U[1] @ V[1].T, a, rtol=0, atol=1e-13 * ref[-1])
