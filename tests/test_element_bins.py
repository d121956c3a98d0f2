"""Host check of the point-location bins (tests/cxx/element_bins_check.cpp
compiled with g++ against salvus_amd/csrc/element_bins.h, the header the
library uses): candidates as complete as a scan over all boxes, in order, and
few enough, also for needle-shaped elements and boxes that are not finite."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_element_bins(tmp_path):
    exe = tmp_path / "element_bins_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", str(ROOT / "salvus_amd" / "csrc"),
                    "-o", str(exe), str(ROOT / "tests" / "cxx" / "element_bins_check.cpp")],
                   check=True, timeout=300)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0, run.stdout[-3000:]
    assert "all bins ok" in run.stdout
