"""Orders of events inside the prefill tiles, replayed on the CPU.

The step loops take these orders from plain headers (csrc/pid_window.h), so a
host program built from the same headers can check every read against every
write without a GPU."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "proxy-attention-lab_amd" / "csrc"


def _run(tmp_path, name: str) -> str:
    exe = tmp_path / name
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", f"-I{CSRC}", str(ROOT / "tests" / "native" / f"{name}.cpp"), "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-4000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, (run.stdout + run.stderr)[-4000:]
    return run.stdout


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_staged_page_entries_outlive_their_readers(tmp_path):
    """A page-id chunk (and its fp8 scales) is overwritten only when every
    wavefront has read the last step that uses it, and is in place before its
    first reader."""
    assert "every entry in place" in _run(tmp_path, "pid_window_driver")
