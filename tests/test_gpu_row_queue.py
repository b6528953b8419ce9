"""The row kernels' queue of kets (buckets by primitive pairs, lanes per ket,
bra primitives split over waves) at its edges, against the quartet-list build
of the same context: one primitive pair only, contraction lengths on both
sides of 32 primitive pairs and beyond the last bucket (24 x 24 = 576), a
handful of kets with long bra loops, and all of these in one molecule.  Both
paths sum the same quartets in FP64 in another order: agreement to 1e-12 of
the largest element."""
import numpy as np
import pytest

from chronusq_public_amd import cqx
from chronusq_public_amd.chem import Molecule

pytestmark = pytest.mark.gpu


def _shells(kinds):
    out = []
    for l, n in kinds:
        out.append(f"{l} {n} 1.00")
        for k in range(n):
            out.append(f"  {0.08 * 2.1 ** k if n > 1 else 0.7:.8f}  {1.0 / (1 + k):.8f}")
    return out


def _basis(h_kinds, o_kinds, natom):
    text = "\n".join(["****", "H 0"] + _shells(h_kinds) + ["****", "O 0"] + _shells(o_kinds) + ["****"]) + "\n"
    Z = [8, 1, 1, 8, 1, 1][:natom]
    xyz = np.array([[0, 0, 0], [0, 1.4, 1.1], [0, -1.4, 1.1], [2.5, 0.4, 3.0], [3.1, 1.9, 4.0], [2.2, -1.2, 4.1]])
    return cqx.BasisSet(text, Molecule(Z, xyz[:natom]))


@pytest.mark.parametrize("h,o,natom", [
    ([("S", 1)], [("S", 1), ("P", 1), ("D", 1)], 3),
    ([("S", 24)], [("S", 24)], 1),
    ([("S", 4), ("S", 1)], [("S", 8), ("P", 5)], 2),
    ([("S", 6), ("P", 1)], [("S", 24), ("S", 9), ("S", 1), ("P", 11), ("P", 3), ("D", 2)], 6)])
@pytest.mark.parametrize("cut", [0.0, 1e-3])
def test_queue_edges(h, o, natom, cut):
    print(f"case: row queue {h} {o} {natom} cut {cut}", flush=True)
    b = _basis(h, o, natom)
    nb = b.nBasis
    rng = np.random.Generator(np.random.PCG64(natom))
    m = rng.normal(size=(nb, nb))
    D = np.asfortranarray(0.5 * (m + m.T))
    tpi = cqx.DirectTPI(b, 1e-12, device=0)
    tpi.set_option("fp32_cut", cut)
    out = []
    for rows in (1, 0):
        tpi.set_option("rows", rows)
        AX = [np.zeros((nb, nb), order="F") for _ in range(2)]
        cqx.GTODirectTPIContraction(tpi).twoBodyContract(
            [cqx.TwoBodyContraction(D, AX[0], True, 0), cqx.TwoBodyContraction(D, AX[1], True, 1)])
        out.append((AX, tpi.last_stats()))
    for key in ("n_quartets", "n_quartets_f32", "n_candidates"):
        assert out[0][1][key] == out[1][1][key], key
    # FP32 quartets lie below the cut, are rounded to about 1e-6 of themselves,
    # and at most nb^2 of them meet in one element
    tol = 1e-12 if cut == 0.0 else 1e-9 * nb * nb
    for x, y in zip(out[0][0], out[1][0]):
        assert np.abs(x - y).max() <= tol * max(1.0, np.abs(y).max())
