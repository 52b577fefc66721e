"""Bounds of the run-time-length transforms (fft_dense.hpp) over every length and
tile, on the CPU."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


@pytest.mark.parametrize("source", ["dense_bounds.cpp", "dense_emulation.cpp"])
def test_every_share_has_a_place(tmp_path, source):
    # a source that no longer compiles is a failure, not a reason to skip
    if shutil.which("hipcc") is None:
        pytest.skip("no hipcc")
    exe = tmp_path / "bounds"
    r = subprocess.run(["hipcc", "-O2", "-std=c++17", "-o", str(exe), os.path.join(ROOT, "tests", "native", source)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "ALL OK" in out.stdout, out.stdout[-2000:]
