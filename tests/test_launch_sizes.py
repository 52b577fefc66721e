"""Blocks that the x passes of run-time row lengths launch.  HIP is replaced by
the test program; no GPU is used."""
import os
import subprocess

from conftest import PKG_DIR, ROOT


def test_run_time_rows_fill_a_round(tmp_path):
    exe = tmp_path / "launch_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "native", "launch_test.cpp"), "-L", PKG_DIR, "-lqsm_gpu",
                    "-Wl,-rpath," + PKG_DIR, "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "ALL OK" in r.stdout, r.stdout[-3000:] + r.stderr[-500:]
