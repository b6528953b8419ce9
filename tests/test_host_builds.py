"""CPU tests of the host side of a build on a HIP runtime without a device
(tests/cpp/fake_hip.cpp: kernels do nothing, streams and events are followed):
a build that fails part way through leaves nothing in flight, and the next one
on the same context starts from tables it has uploaded itself; the times of a
call's contraction groups add up."""
import ctypes as C
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CASES = ["nothing_in_flight", "tables_after_failure", "groups_add_up"]


def _cont(cqx, np, nb, n):
    D = np.asfortranarray(np.eye(nb))
    return [cqx.TwoBodyContraction(D, np.zeros((nb, nb), order="F"), True, t) for t in ([0, 1] * n)[:n]]


def _contract(cqx, np, tpi, n=2):
    """None, or the error of the build"""
    try:
        cqx.GTODirectTPIContraction(tpi).twoBodyContract(_cont(cqx, np, tpi.basis.nBasis, n), False)
    except cqx.CErr as e:
        return str(e)


def _child(fakelib, case):
    fake = C.CDLL(fakelib, mode=C.RTLD_GLOBAL)
    fake.fake_in_flight.restype = fake.fake_unwritten_tables.restype = C.c_longlong
    import numpy as np
    from chronusq_public_amd import cqx
    from chronusq_public_amd.chem import cluster_box, water_cluster

    def tpi_of(n=1):
        return cqx.DirectTPI(cqx.BasisSet("6-31G(d)", water_cluster(n, cluster_box(n), 1)), 1e-12)

    def read_back(w):
        fake.fake_read_back(C.c_longlong(w))

    def failing(run):
        """run() with the first, second, ... allocation failing, until none does"""
        k, errors = 0, 0
        while True:
            k += 1
            fake.fake_fail_malloc(C.c_longlong(k))
            e = run(k)
            fake.fake_fail_malloc(C.c_longlong(0))
            if e is None:
                assert errors > 0
                return
            assert "out of memory" in e, e
            errors += 1

    if case == "nothing_in_flight":
        def run(k):
            tpi = fresh[k]
            e = _contract(cqx, np, tpi)
            assert fake.fake_in_flight() == 0, (k, e, fake.fake_in_flight())
            return e
        for word, rows in ((0, 1), (5, 1), (5, 0)):
            fresh = [tpi_of(2) for _ in range(80)]
            for t in fresh:
                t.set_option("rows", rows)
                t.set_option("list_cap", 1 << 28 if word == 0 else 1000)
            read_back(word)
            failing(run)
            read_back(0)
    elif case == "tables_after_failure":
        def run(k):
            tpi = tpi_of()
            tpi.set_option("rows", 0)  # lists for every class pair, none with a candidate
            assert _contract(cqx, np, tpi) is None
            tpi.set_option("rows", 1)  # a small build: its tables are kept
            assert _contract(cqx, np, tpi) is None
            tpi.set_option("rows", 0)  # every list with candidates: larger tables
            fake.fake_fail_malloc(C.c_longlong(k))
            read_back(5)
            e = _contract(cqx, np, tpi)
            read_back(0)
            fake.fake_fail_malloc(C.c_longlong(0))
            tpi.set_option("rows", 1)
            assert _contract(cqx, np, tpi) is None
            assert fake.fake_unwritten_tables() == 0, (k, e)
            return e

        k = 0
        while run(k := k + 1) is not None:
            pass
        assert k > 1
    else:
        tpi = tpi_of()
        for n, groups in ((2, 1), (8, 1), (9, 2), (20, 3)):
            assert _contract(cqx, np, tpi, n) is None
            assert tpi.last_stats()["ms_eri"] == groups  # every interval lasts 1 ms
    print("child ok")


@pytest.fixture(scope="module")
def fakelib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                        "-I", "/opt/rocm/include", os.path.join(HERE, "cpp", "fake_hip.cpp"), "-o", out],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("case", CASES)
def test_host_side(fakelib, case):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fakelib, case], capture_output=True, text=True,
                       timeout=120, cwd=os.path.dirname(HERE))
    assert r.returncode == 0 and "child ok" in r.stdout, r.stdout + r.stderr


if __name__ == "__main__":
    sys.path.insert(0, os.path.dirname(HERE))
    _child(*sys.argv[1:])
