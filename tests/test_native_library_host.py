"""Building the operators' native library (libtokserve_torch.so) beside the C library (CPU)."""

import subprocess
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "tokserve_amd" / "csrc"


def test_make_without_a_torch_builds_the_c_library_alone() -> None:
    run = subprocess.run(["make", "-n", "-C", CSRC, "PYTHON=false"], capture_output=True, text=True)
    assert run.returncode == 0, run.stderr
    assert "torch" not in run.stdout


def test_make_notices_another_torch(tmp_path) -> None:
    stamp = tmp_path / "torch_id"

    def make() -> int:
        subprocess.run(["make", "-C", CSRC, f"PYTHON={sys.executable}", f"BUILD={tmp_path}", stamp],
                       check=True, capture_output=True)
        return stamp.stat().st_mtime_ns

    first = make()
    assert torch.__version__ in stamp.read_text()
    assert make() == first
    stamp.write_text(stamp.read_text().replace(torch.__version__, "1.0.0"))
    written = stamp.stat().st_mtime_ns
    assert make() > written
