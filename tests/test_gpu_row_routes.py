"""Options that send classes to the generic kernel, which has FP64 only: such
classes keep it with row kernels on, so the quartets evaluated in FP32 are the
quartet-list build's, and the sums agree (FP64 to 1e-12 of the largest element;
the FP32 quartets, rounded to about 1e-6 of themselves, at most nb^2 of them in
one element: 1e-6 of the largest integral times that)."""
import numpy as np
import pytest

from chronusq_public_amd import cqx
from chronusq_public_amd.chem import cluster_box, water_cluster

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opts", [{"fast_max_nc": 9}, {"fast_max_nc": 20}, {"use_wave": 0},
                                  {"fast_max_nc": 9, "use_wave": 0}, {"fast_max_nc": 0}, {}])
@pytest.mark.parametrize("cut", [0.0, 1.0])
def test_generic_classes_stay_generic(opts, cut):
    print(f"case: row routes {opts} cut {cut}", flush=True)
    tpi = cqx.DirectTPI(cqx.BasisSet("cc-pVDZ", water_cluster(2, cluster_box(2), 4)), 1e-12, device=0)
    for k, v in dict(opts, fp32_cut=cut).items():
        tpi.set_option(k, v)
    nb = tpi.basis.nBasis
    rng = np.random.Generator(np.random.PCG64(8))
    D = rng.normal(size=(nb, nb)) / np.sqrt(nb)
    D = np.asfortranarray(0.5 * (D + D.T))
    out = []
    for rows in (1, 0):
        tpi.set_option("rows", rows)
        AX = [np.zeros((nb, nb), order="F") for _ in range(2)]
        cqx.GTODirectTPIContraction(tpi).twoBodyContract(
            [cqx.TwoBodyContraction(D, AX[t], True, t) for t in (0, 1)])
        out.append((AX, tpi.last_stats()))
    for key in ("n_quartets", "n_quartets_f32", "n_candidates", "n_prim_quartets_max"):
        assert out[0][1][key] == out[1][1][key], key
    tol = 1e-12 if cut == 0.0 else 1e-6 * nb * nb
    for x, y in zip(out[0][0], out[1][0]):
        assert np.abs(x - y).max() <= tol * max(1.0, np.abs(y).max())
