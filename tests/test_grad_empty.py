"""CPU test of the templated gradient kernels (csrc/eri_grad_impl.hpp) on an
emulated block: a quartet without primitive pairs adds nothing."""
import os
import subprocess

from conftest import ROOT


def test_empty_quartets_add_nothing(tmp_path):
    exe, cpp = str(tmp_path / "grad_test"), os.path.join(ROOT, "tests", "cpp")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wno-attributes", "-Wno-unknown-pragmas",
                        "-I", os.path.join(cpp, "wave"), "-I", os.path.join(ROOT, "chronusq_public_amd", "csrc"),
                        os.path.join(cpp, "grad_test.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout)
    assert r.stdout.count(" ok ") == 3
