"""CPU test of the staged J/K digestion (csrc/digest_staged.hpp) on an emulated
wave: quartets of two molecules of different sizes in one wave, in both orders,
every plane followed by a page that may not be touched."""
import os
import subprocess

from conftest import ROOT


def test_staged_digestion_stays_in_its_molecules_planes(tmp_path):
    exe, cpp = str(tmp_path / "staged_test"), os.path.join(ROOT, "tests", "cpp")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wno-attributes", "-Wno-unknown-pragmas",
                        "-I", os.path.join(cpp, "wave"), "-I", os.path.join(ROOT, "chronusq_public_amd", "csrc"),
                        os.path.join(cpp, "staged_test.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout)
    assert r.stdout.count(" ok ") == 14
