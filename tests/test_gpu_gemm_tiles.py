"""The tile of a grouped GEMM launch does not change its results: the 64 x 64
default of small launches and the 128 x 128 tiles of large ones agree to the
bit (the K split follows from the problem alone and k is summed in order)."""
import numpy as np
import pytest

from oracle import heff as oheff
from su2dmrg_amd import synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from su2dmrg_amd import lib as L
    c = L.Context(0)
    yield c
    c.close()


# tile edges (63, 64, 65, 127, 129), one-element sectors, and depths on both
# sides of the shortest split (128 and 256 deep)
@pytest.mark.parametrize("dims,nterm", [
    ((1, 2, 1), 1),
    ((63, 65, 64), 2),
    ((127, 129, 16), 3),
    ((128, 257, 241), 2),
])
@pytest.mark.parametrize("bits,big,rtol", [(64, 1, 1e-10), (32, 0, 5e-5)])
def test_default_tiles_match_large_tiles_bitwise(ctx, dims, nterm, bits, big, rtol):
    from su2dmrg_amd import lib as L
    print(f"tiles dims={dims} nterm={nterm} bits={bits}", flush=True)
    work = synthetic.small(seed=5, twoj=(1, 3, 5), dims=dims, nterm=nterm)
    dev = L.upload_workload(ctx, work)
    plan = dev["plan"]
    plan.set_precision(bits)
    plan.apply(dev["psi"], dev["out"])
    a = dev["out"].download()
    plan.set_variants(big, big)
    plan.apply(dev["psi"], dev["out"])
    assert np.array_equal(a, dev["out"].download())
    ref = oheff.heff_apply(work["psi"], work["hl"], work["hr"], work["terms"])
    got = L.unpack_wavefunction(dev["out"], a)
    num = sum(float(np.sum((got[j] - ref[j]) ** 2)) for j in ref)
    den = sum(float(np.sum(ref[j] ** 2)) for j in ref)
    assert np.sqrt(num / den) < rtol
