"""The digest that kernel profiles record changes with everything the ERI and
digestion kernels are built from: each local file they include, however
indirectly, and the Rys tables the build derives."""
import os
import re
import shutil

import pytest

from chronusq_public_amd import build


def _included():
    todo = [f for f in os.listdir(build.CSRC) if re.match(r"(eri_|front|kernels).*\.hip$", f)]
    seen = set()
    while todo:
        f = todo.pop()
        if f in seen or not os.path.exists(os.path.join(build.CSRC, f)):
            continue
        seen.add(f)
        with open(os.path.join(build.CSRC, f)) as fh:
            todo += re.findall(r'#include "([^"]+)"', fh.read())
    return sorted(f for f in seen if not f.endswith("_data.inc"))


def test_every_included_file(tmp_path, monkeypatch):
    csrc = str(tmp_path / "csrc")
    shutil.copytree(build.CSRC, csrc)
    monkeypatch.setattr(build, "CSRC", csrc)
    before, files = build.source_digest(), _included()
    assert "screen.hpp" in files and "rys.hpp" in files
    for f in files:
        path = os.path.join(csrc, f)
        with open(path, "rb") as fh:
            text = fh.read()
        with open(path, "wb") as fh:
            fh.write(text + b"\n")
        assert build.source_digest() != before, f
        with open(path, "wb") as fh:
            fh.write(text)
    assert build.source_digest() == before


@pytest.mark.parametrize("name", ["rys_powers", "rys_halves"])
def test_derived_tables(monkeypatch, name):
    before, derive = build.source_digest(), getattr(build, name)
    monkeypatch.setattr(build, name, lambda *a: derive(*a) * 1.0000001)
    assert build.source_digest() != before
