"""Lanczos vector algebra for more jobs than one launch carries, with vectors
on both sides of every size at which the kernels change (one workgroup with
4, 8 and 16 elements a thread, then a grid per dependent sum): every run of
the batch equals itself alone, bit for bit, and reaches the ground energy."""
import numpy as np
import pytest

from oracle import dmrg as od
from oracle import ed

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


# (lx, ly, D): vectors of a few elements up to about 50000
@pytest.mark.parametrize("specs", [
    [(4, 2, 20)] * 17 + [(6, 2, 70)],
    [(3, 4, 40), (4, 4, 70), (4, 4, 110), (6, 4, 150), (6, 4, 280)],
])
def test_mixed_lengths_in_one_batch(ctx, specs):
    from su2dmrg_amd import lib as L
    print(f"krylov batch {specs}", flush=True)

    def new(lx, ly, d):
        return L.Dmrg(ctx, lx, ly, 2.0, 0.0, 2, 0, d)

    alone = {}
    for s in sorted(set(specs)):
        g = new(*s)
        g.warmup()
        g.sweep()
        g.sweep()
        alone[s] = np.array(g.energies())
        g.close()
    b = L.Batch(ctx)
    runs = [(s, new(*s)) for s in specs]
    for s, g in runs:
        b.add(g, [(s[2], 64)] * 2)
    while b.tick() > 0:
        pass
    for s, g in runs:
        assert np.array_equal(np.array(g.energies()), alone[s]), s
    b.close()
    for _, g in runs:
        g.close()
    for s in set(specs):
        if s in ((4, 2, 20), (6, 2, 70)):   # untruncated
            e = ed.ground_energy(od.Lattice(s[0], s[1], jcoup=2.0, bdry=2), 0)
            assert abs(alone[s][-1] - e) < 1e-8 * abs(e)
