"""Host check of the colour launches' node numbering (tests/cxx/
colour_tiles_check.cpp, compiled for the host with the library's tiles.cpp):
the words that the tables by kinds of tiles give are those of a numbering made
node by node."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_colour_tiles(tmp_path):
    exe = tmp_path / "colour_tiles_check"
    src = ROOT / "salvus_amd" / "csrc"
    subprocess.run(["hipcc", "--offload-host-only", "-x", "hip", "-O1", "-std=c++17", "-I", str(src), "-o", str(exe),
                    str(ROOT / "tests" / "cxx" / "colour_tiles_check.cpp"), str(src / "tiles.cpp")],
                   check=True, timeout=300)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0, run.stdout[-3000:]
    assert "boxes alike" in run.stdout
