"""Run-time axis lengths up to 512 (fft_dense.hpp): the index functions of the
register and matrix-core stages on the CPU, and the dipole operator on axes at
the edges of the dense radices' tiles on the GPU, against the f64 oracle."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_dense_stages_cpu_emulation(tmp_path):
    exe = tmp_path / "dense_emu"
    r = subprocess.run(["hipcc", "-O2", "-std=c++17", "-o", str(exe),
                        os.path.join(ROOT, "tests", "native", "dense_emulation.cpp")],
                       capture_output=True, text=True)
    if r.returncode != 0:
        pytest.skip("hipcc unavailable: " + r.stderr[-300:])
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and "ALL OK" in out.stdout, out.stdout[-2000:]


# 17 and 31: one row tile, first and last of its rows; 34 and 61: two; 97: four;
# 251: eight; 2 p, 3 p, 5 p: a register stage after the dense one; 289 and 323:
# two dense stages; 262, 502, 511: tiles of 8 columns; 243, 250: register
# radices only; 257: chirp-z, beside a dense axis
@pytest.mark.gpu
@pytest.mark.parametrize("n", [17, 31, 34, 61, 82, 97, 123, 164, 205, 243, 250, 251, 254, 257, 262, 289, 323,
                               502, 511])
def test_dipole_dense_axis(qsm, oracle, n):
    # the largest error of a transform of these lengths in FP32 is below
    # 4e-7 of its largest output (CPU emulation); six transforms, and the
    # field's maximum is below the susceptibility's
    for axis in range(3):
        dims = [6, 9, 10]
        dims[axis] = n
        rng = np.random.default_rng(n * 3 + axis)
        chi = rng.standard_normal(int(np.prod(dims)))
        vs, b = (0.9, 1.1, 1.3), (0.2, -0.1, 1.0)
        f = qsm.dipole_forward(chi, qsm.Grid(tuple(dims), vs), b)
        ref = oracle.dipole_forward(chi, tuple(dims), vs, b)
        assert np.max(np.abs(f - ref)) < 6 * 4e-7 * np.max(np.abs(chi)) * 2
