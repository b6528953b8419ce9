"""Gradient contractions whose primitive pairs are screened out (option
prim_screen) add nothing to the outputs, in every templated and generic class."""
import numpy as np
import pytest

from chronusq_public_amd import cqx
from chronusq_public_amd.chem import cluster_box, water_cluster

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis", ["cc-pVDZ", "cc-pVTZ"])
def test_gradient_without_primitive_pairs(basis):
    print(f"case: gradient without primitive pairs, {basis}", flush=True)
    mol = water_cluster(1, cluster_box(1), 2)
    tpi = cqx.DirectTPI(cqx.BasisSet(basis, mol), 1e-12, device=0)
    nb, ng = tpi.basis.nBasis, 3 * mol.natom
    rng = np.random.Generator(np.random.PCG64(2))
    D = rng.normal(size=(nb, nb))
    D = np.asfortranarray(D + D.T)

    def run():
        out = [[cqx.TwoBodyContraction(D, np.zeros((nb, nb), order="F"), True, t) for t in (0, 1)] for _ in range(ng)]
        cqx.DirectGradContraction(tpi).gradTwoBodyContract(out)
        return np.array([c.AX for g in out for c in g])

    full = run()  # leaves its derivative sums behind
    assert np.abs(full).max() > 0.0
    tpi.set_option("prim_screen", 1e300)
    assert np.abs(run()).max() == 0.0
    tpi.set_option("prim_screen", 1e-18)
    assert np.abs(run() - full).max() <= 1e-12 * np.abs(full).max()
