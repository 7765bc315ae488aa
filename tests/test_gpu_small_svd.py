"""Sector blocks small enough for one CU's LDS (and the first ones that are not) against LAPACK.

The lanes per pair change at 32 and 64 columns, the compiled unrollings every 32, 16 or 16 rows,
the LDS limit lies near 96 x 96 and the row limit at 128; both orientations, odd and even column
counts, rank-deficient and zero blocks.
"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (1, 7), (2, 2), (3, 2), (5, 16), (17, 16), (32, 32), (33, 32), (33, 33), (48, 37),
          (64, 64), (65, 64), (66, 65), (81, 80), (96, 96), (97, 96), (128, 3), (128, 70),
          (129, 20), (99, 99)]


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("rank", ["full", "deficient"])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_small_block_against_lapack(ctx, rows, cols, rank):
    # The rotations applied to a column (under 10 sweeps of k - 1) each leave eps of its norm:
    # 10 k eps = 1.4e-13 at k = 128; 5e-13 bounds the orthonormal side and, times s_max, the values
    # and the reconstruction.
    from su2dmrg_amd import lib as L
    for m, n in {(rows, cols), (cols, rows)}:
        print(f"small svd {m}x{n} {rank}", flush=True)
        sys.stdout.flush()
        rng = np.random.default_rng(1000 * m + n)
        k = min(m, n)
        u, _ = np.linalg.qr(rng.standard_normal((m, k)))
        v, _ = np.linalg.qr(rng.standard_normal((n, k)))
        s = np.logspace(0, -9, k)
        if rank == "deficient":
            s[(2 * k) // 3:] = 0.0
            s[0] = 1.0
        a = (u * s) @ v.T
        # a second sector of exact zeros and a third of one column share the launch
        b = rng.standard_normal((4, 1))
        t = L.wavefunction(ctx, [1, 3, 5], [m, 6, 4], [n, 5, 1],
                           {1: a, 3: np.zeros((6, 5)), 5: b})
        # the short side is the orthonormal one
        p1, p2 = (1.0, 0.0) if m >= n else (0.0, 1.0)
        # one column less than there are (the zero sector keeps none): a cut is possible
        U, V, kept, _ = L.svd_truncate(ctx, t, p1, p2, k + 5)
        ref = np.linalg.svd(a, compute_uv=False)
        got = np.sort(np.linalg.norm(U[1] if m >= n else V[1], axis=0))[::-1]
        top = ref[0]
        np.testing.assert_allclose(got, ref[:got.size], rtol=0, atol=5e-13 * top)
        np.testing.assert_allclose(U[1] @ V[1].T, a, rtol=0, atol=5e-13 * top)
        q = V[1] if m >= n else U[1]
        np.testing.assert_allclose(q.T @ q, np.eye(q.shape[1]), rtol=0, atol=5e-13)
        assert 3 not in U
        np.testing.assert_allclose(U[5] @ V[5].T, b, rtol=0, atol=1e-14)
        assert abs(kept[-1] - np.linalg.norm(b)) < 1e-14 * np.linalg.norm(b) + 1e-15
