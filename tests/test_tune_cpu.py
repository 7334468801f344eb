"""The autotuner's choice among candidates, on planted timings: a slow start
and noise must not hide that the first candidate is 6 % faster than the next."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_choice_on_planted_timings(tmp_path):
    exe = str(tmp_path / "harness")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I" + os.path.join(ROOT, "nektar_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpu_tune", "harness.cpp"), "-o", exe], check=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout
