"""The ring of LDS buffers that kernels fill by counted DMA (csrc/kernels/lds_stages.h), run on the host against a model of the queue
of moves: every block has landed when it is read, for every number of buffers, moves and blocks."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.timeout(120)
def test_blocks_have_landed_when_they_are_read(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host compiler")
    exe = tmp_path / "lds_stages_selftest"
    r = subprocess.run([cxx, "-std=c++17", "-O1", str(ROOT / "csrc/tests/lds_stages_selftest.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "lds_stages OK" in r.stdout, r.stdout + r.stderr
