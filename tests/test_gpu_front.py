"""Front and back of a build (norms, planes, candidates, transforms back, one
launch each) where they can go wrong: device matrices read and added to in
place against staged host ones, outputs that share memory, and small builds,
whose quartet lists are launched over their capacity without reading counts
back, against the same build with its lists in counted batches.

The same quartets are summed in FP64 in another order: agreement to 1e-12 of
the largest element (mixed precision: the same quartets go to FP32 and are
rounded alike, their sums differ in order only)."""
import numpy as np
import pytest

from chronusq_public_amd import cqx
from chronusq_public_amd.chem import cluster_box, water_cluster

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _tpi(basis, n, **opts):
    tpi = cqx.DirectTPI(cqx.BasisSet(basis, water_cluster(n, cluster_box(n), 5)), 1e-12)
    for k, v in opts.items():
        tpi.set_option(k, v)
    return tpi


def _mat(rng, nb, cplx, her):
    m = rng.normal(size=(nb, nb)) + (1j * rng.normal(size=(nb, nb)) if cplx else 0)
    return np.asfortranarray((0.5 * (m + m.conj().T) if her else m) / np.sqrt(nb))


def _host(tpi, cont, A0, screen=True):
    out = [np.array(a, order="F") for a in A0]
    cqx.GTODirectTPIContraction(tpi).twoBodyContract(
        [cqx.TwoBodyContraction(X, a, her, typ) for (X, typ, her), a in zip(cont, out)], screen)
    return out, tpi.last_stats()


def _close(a, b):
    for x, y in zip(a, b):
        assert np.abs(x - y).max() <= TOL * max(1.0, np.abs(y).max())


@pytest.mark.parametrize("basis,n,cplx,screen", [("sto-3g", 1, False, True), ("6-31G(d)", 2, True, True),
                                                 ("cc-pVTZ", 1, False, False), ("cc-pVDZ", 9, True, True)])
def test_in_place_device_matrices_equal_host_ones(basis, n, cplx, screen):
    tpi = _tpi(basis, n)
    nb = tpi.basis.nBasis
    rng = np.random.Generator(np.random.PCG64(n))
    kinds = [(0, True), (1, True), (1, False), (0, False), (1, True)]
    cont = [(_mat(rng, nb, cplx, her), typ, her) for typ, her in kinds]
    A0 = [_mat(rng, nb, cplx, True) for _ in cont]
    want, st = _host(tpi, cont, A0, screen)
    dA = [cqx.DeviceMatrix(tpi, nb, cplx).upload(a) for a in A0]
    dX = [cqx.DeviceMatrix(tpi, nb, cplx).upload(c[0]) for c in cont]
    cqx.GTODirectTPIContraction(tpi).twoBodyContract(
        [cqx.TwoBodyContraction(x, a, c[2], c[1]) for x, a, c in zip(dX, dA, cont)], screen)
    assert tpi.last_stats()["n_quartets"] == st["n_quartets"]
    assert tpi.last_stats()["n_candidates"] == st["n_candidates"]
    _close([a.download() for a in dA], want)


@pytest.mark.parametrize("noalloc", [False, True])
def test_outputs_that_share_memory(noalloc):
    """A shared output keeps its last contraction's sum (each adds to a copy),
    in the allocation-free call the sum of all (added one after the other)."""
    tpi = _tpi("6-31G(d)", 2)
    nb = tpi.basis.nBasis
    rng = np.random.Generator(np.random.PCG64(4))
    cont = [(_mat(rng, nb, False, True), typ, True) for typ in (0, 1, 1)]
    A0 = _mat(rng, nb, False, True)
    parts, _ = _host(tpi, cont, [np.zeros_like(A0)] * 3)
    dA = cqx.DeviceMatrix(tpi, nb, False).upload(A0)
    lst = [cqx.TwoBodyContraction(cqx.DeviceMatrix(tpi, nb, False).upload(c[0]), dA, c[2], c[1]) for c in cont]
    gto = cqx.GTODirectTPIContraction(tpi)
    (gto.twoBodyContractNoAlloc if noalloc else gto.twoBodyContract)(lst)
    _close([dA.download()], [A0 + (sum(parts) if noalloc else parts[-1])])


@pytest.mark.parametrize("basis,n,cut", [("cc-pVDZ", 1, 0.0), ("cc-pVDZ", 2, 1e-4), ("cc-pVTZ", 1, 0.0)])
def test_small_builds_equal_counted_ones(basis, n, cut):
    a, b = _tpi(basis, n, fp32_cut=cut), _tpi(basis, n, fp32_cut=cut, list_cap=16)
    nb = a.basis.nBasis
    rng = np.random.Generator(np.random.PCG64(6))
    cont = [(_mat(rng, nb, False, True), typ, True) for typ in (0, 1)]
    for _ in range(2):  # the second build finds its tables in place
        x, sa = _host(a, cont, [np.zeros((nb, nb))] * 2)
        y, sb = _host(b, cont, [np.zeros((nb, nb))] * 2)
        for key in ("n_quartets", "n_quartets_f32", "n_candidates", "n_prim_quartets_max"):
            assert sa[key] == sb[key], key
        _close(x, y)
        cont = [(1e-3 * X, typ, her) for X, typ, her in cont]  # fewer candidates
