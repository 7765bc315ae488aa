"""Environment scatters at the block size where a workgroup's share of a block changes (2^16
elements): one element row below, at and above it, against the oracle, on the enlarged basis."""
import numpy as np
import pytest

from oracle import dmrg as od
from oracle.su2 import Bond
from test_gpu_env import RTOL, _blocks, _rel, _scalar

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("left", [True, False])
@pytest.mark.parametrize("dims", [(255, 257), (256, 256), (1, 300)])
def test_scatter_around_the_long_chunks(ctx, left, dims):
    from su2dmrg_amd import lib as L
    from su2dmrg_amd import synthetic
    print(f"env chunks left={left} dims={dims}", flush=True)
    twoj = [0, 2]
    rng = np.random.default_rng(sum(dims) + int(left))
    E = od.Enlarged(Bond(twoj, list(dims)), left)
    pos = dict(zip(twoj, dims))
    H = {j: (lambda m: m + m.T)(rng.standard_normal((d, d))) for j, d in pos.items()}
    S = {(a, b): rng.standard_normal((pos[a], pos[b])) for a, b in synthetic.transitions(twoj)}
    dH = _scalar(ctx, L, twoj, list(dims), H)
    dS = L.vector_operator(ctx, twoj, list(dims), S)
    for kind, op, ref, nleg in (
            ("overlap", dH, od.enlarge(E, H, {}, [], left)[0], 2),
            ("pairup", dS, od.enlarge(E, None, {}, [(0.7, S)], left)[0], 2),
            ("op_transform", dS, od.enlarge(E, None, {0: S}, [], left)[1][0], 3),
            ("initial", None, od.enlarge(E, None, {}, [], left)[2], 3)):
        if nleg == 2:
            ref = {(j, j): b for j, b in ref.items()}
        got = _blocks(L.env_transform(ctx, kind, left, twoj, list(dims), None, op, 0.7), nleg)
        assert _rel(got, ref) < RTOL, kind
