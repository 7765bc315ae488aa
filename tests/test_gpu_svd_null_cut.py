"""A cut inside the null space: sectors of equal norm keep the same fraction of their null
directions, whichever kernel their size sends them to."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


# on both sides of one compute unit's LDS (96 columns, 128 rows) and of 256 columns
SIZES = [(40, 44), (92, 90), (130, 120), (210, 200), (300, 310), (640, 600)]


@pytest.mark.parametrize("tail", [False, True])
@pytest.mark.parametrize("frac", [0.25, 0.5, 0.8])
def test_null_directions_by_size(ctx, frac, tail):
    from su2dmrg_amd import lib as L
    print(f"null cut at {frac}, tail={tail}", flush=True)
    rng = np.random.default_rng(7)
    psi, nulls, cols = {}, {}, 0
    for i, (m, n) in enumerate(SIZES):
        k = min(m, n)
        u, _ = np.linalg.qr(rng.standard_normal((m, k)))
        v, _ = np.linalg.qr(rng.standard_normal((n, k)))
        x = np.arange(k) / k
        s = np.where(x < 0.6, 10.0 ** (-2.5 * x / 0.6), 0.0)
        if tail:   # down to 1e-10 before the null space
            s = np.where((x >= 0.6) & (x < 0.75), 10.0 ** (-2.5 - 50 * (x - 0.6)), s)
        psi[2 * i + 1] = (u * (s / np.linalg.norm(s))) @ v.T
        nulls[2 * i + 1] = int(np.sum(s == 0))
        cols += k
    twoj = sorted(psi)
    t = L.wavefunction(ctx, twoj, [m for m, _ in SIZES], [n for _, n in SIZES], psi)
    total = sum(nulls.values())
    take = int(frac * total)
    U, V, kept, _ = L.svd_truncate(ctx, t, 1.0, 0.0, cols - total + take)
    for (m, n), j in zip(SIZES, twoj):
        got = U[j].shape[1] - (min(m, n) - nulls[j])
        # the levels of all sectors interleave: at most one off the common fraction each
        assert abs(got - nulls[j] * take / total) <= 1.5, (m, n, got, nulls[j])
    kept = np.array(kept)
    assert np.sum(kept < 1e-13) == take   # reported as computed
