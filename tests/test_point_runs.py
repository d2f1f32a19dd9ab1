"""The length of a point set's planar runs, as beep_hip_set_geometry reads it
from the first patches (tests/point_runs_check.cpp, on the CPU): points whose
normal is not a number end a run and never stop the search."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_shortest_normal_run(tmp_path):
    exe = tmp_path / "point_runs_check"
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'beep3_amd' / 'csrc'}",
                    str(ROOT / "tests" / "point_runs_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=20)
    assert r.stdout.split() == ["12", "24", "1", "1", "1"]
