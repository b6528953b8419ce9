"""bench.py keeps the figures of its finished legs when a later one dies: the
line is printed with the error, nothing further is started, and the exit status
is not zero (CPU; the measured workload is replaced by fixed numbers)."""
import json
import subprocess
import sys
import types

import numpy as np
import pytest

import bench


class _Build:
    def __init__(self, *a, **k):
        self.mol = self.gbs = self.gto = None
        self.mats, self.types, self.cplx = [], [], False
        self.basis = types.SimpleNamespace(nBasis=1)
        self.tpi = types.SimpleNamespace(
            set_option=lambda *a: None,
            last_stats=lambda: {"n_quartets": 1, "n_candidates": 1, "n_prim_quartets_max": 1})

    def timed(self, steps, warmup):
        return 2.0, 1.0, 1e9, 0.0

    def outputs(self):
        return [np.zeros((1, 1))]


def _run(monkeypatch, capsys, programs):
    """The printed line and the exit status, legs run as the given programs."""
    started = []

    def command(name, size):
        started.append(name)
        return [sys.executable, "-c", programs[name]]

    monkeypatch.setattr(bench, "Build", _Build)
    monkeypatch.setattr(bench, "leg_command", command)
    monkeypatch.setattr(bench, "profile_counters", lambda w: None)
    monkeypatch.setattr(sys, "argv", ["bench.py", "--steps", "4", "--no-cpu", "--no-host", "--no-graph"])
    status = 0
    try:
        bench.main()
    except SystemExit as e:
        status = e.code
    out = capsys.readouterr().out.strip().splitlines()
    assert len(out) == 1
    return json.loads(out[0]), status, started


FINE = "print('note'); print('{\"x\": 1}')"


def test_all_legs(monkeypatch, capsys):
    line, status, started = _run(monkeypatch, capsys, dict(mixed=FINE, batched=FINE, serving=FINE))
    assert status == 0 and line["value"] == 2.0 and started == ["mixed", "batched", "serving"]
    assert all(line[k] == {"x": 1} for k in started)


@pytest.mark.parametrize("dies", ["batched", "serving"])
def test_a_leg_that_dies(monkeypatch, capsys, dies):
    programs = dict(mixed=FINE, batched=FINE, serving=FINE)
    programs[dies] = "import os; os.abort()"
    line, status, started = _run(monkeypatch, capsys, programs)
    assert status == 1 and started[-1] == dies
    assert line["value"] == 2.0 and line["mixed"] == {"x": 1}
    assert "-6" in line[dies]["error"]


def test_a_leg_without_end():
    assert "within" in bench.child_leg([sys.executable, "-c", "import time; time.sleep(60)"], timeout=1)["error"]


def test_leg_command_is_the_leg():
    cmd = bench.leg_command("mixed", 3)
    r = subprocess.run(cmd[:2] + ["--help"], capture_output=True, text=True)
    assert r.returncode == 0 and "--leg" in r.stdout and cmd[2:5] == ["--leg", "mixed", "3"]
