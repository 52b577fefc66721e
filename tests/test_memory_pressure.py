"""The library where memory runs out: what it keeps between calls is given back
before a call of its own fails on the device, and a host allocation that fails
while a table is formed leaves no part of it behind.  HIP is replaced by the
test program; no GPU is used."""
import os
import subprocess

import pytest

from conftest import PKG_DIR, ROOT


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("memory") / "memory_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "native", "memory_test.cpp"), "-L", PKG_DIR, "-lqsm_gpu",
                    "-Wl,-rpath," + PKG_DIR, "-o", str(out)], check=True)
    return str(out)


def _run(exe, *args):
    r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "ALL OK" in r.stdout, r.stdout[-2000:] + r.stderr[-500:]
    return r.stdout


def test_kept_memory_is_given_back_to_own_calls(exe):
    _run(exe, "device")


def test_failed_host_allocations_stay_inside(exe):
    _run(exe, "host")


# The allocations of a call come in this order: the volume's descriptor and
# tables one axis at a time, each table growing in steps; 40 covers them all
# for the shortest length and the tables of the longest.
def test_table_whole_after_failed_allocation(exe):
    want = _run(exe, "tables", "0")
    for k in range(1, 41):
        assert _run(exe, "tables", str(k)) == want, k
