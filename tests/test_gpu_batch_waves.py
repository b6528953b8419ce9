"""Batches whose wave kernels take two quartets a wave above 216 components
((dp|dp), (dd|pp): lists of at least 8192 quartets), so that a wave may hold
quartets of two molecules: the larger molecule first, the smallest last, against
each molecule alone.  The same quartets are summed in FP64 in another order:
1e-12 of the largest element; in mixed precision the FP32 quartets, each below
fp32_cut = 1e-4 with a relative rounding below 1e-6, may be summed in another
order too: 1e-9."""
import numpy as np
import pytest

from chronusq_public_amd import cqx
from chronusq_public_amd.chem import cluster_box, water_cluster

pytestmark = pytest.mark.gpu


def _contract(tpi, dens, her):
    out = []
    for D in dens:
        for typ in (0, 1):
            out.append(cqx.TwoBodyContraction(D, np.zeros_like(D, order="F"), her, typ))
    cqx.GTODirectTPIContraction(tpi).twoBodyContract(out)
    return [c.AX for c in out], tpi.last_stats()


@pytest.mark.parametrize("sizes", [(12, 2, 1), (1, 2, 12)])
@pytest.mark.parametrize("her,cut", [(True, 0.0), (True, 1e-4), (False, 0.0)])
def test_waves_of_two_molecules(sizes, her, cut):
    print(f"case: waves of two molecules, sizes {sizes} her {her} cut {cut}", flush=True)
    parts = [cqx.BasisSet("cc-pVDZ", water_cluster(n, cluster_box(n), 3)) for n in sizes]
    rng = np.random.Generator(np.random.PCG64(12))
    dens = []
    for b in parts:
        m = rng.normal(size=(b.nBasis, b.nBasis)) / np.sqrt(b.nBasis)
        dens.append(np.asfortranarray(0.5 * (m + m.T) if her else m))
    alone, nq = [], 0
    for b, D in zip(parts, dens):
        tpi = cqx.DirectTPI(b, 1e-12, device=0)
        tpi.set_option("fp32_cut", cut)
        AX, st = _contract(tpi, [D], her)
        alone += AX
        nq += st["n_quartets"]
    tpi = cqx.DirectTPI(cqx.BasisSet.batch(parts), 1e-12, device=0)
    tpi.set_option("fp32_cut", cut)
    got, st = _contract(tpi, dens, her)
    assert st["n_quartets"] == nq
    for x, y in zip(got, alone):
        assert np.abs(x - y).max() <= (1e-9 if cut else 1e-12) * np.abs(y).max()
