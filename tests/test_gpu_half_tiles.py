"""Column passes of run-time lengths in tiles of 8 columns (half tiles), at the
edges of the lengths that take them, against the f64 oracle."""
import numpy as np
import pytest

from conftest import nrmse_dc

pytestmark = pytest.mark.gpu


# 127, 129: just outside (129 = 3 x 43); 130, 252: register radices, the first
# and the last of the range; 136, 153, 221, 255: one dense radix of one row
# tile; 164, 205: of two; 212: of four, 4 butterflies a column
@pytest.mark.parametrize("n", [127, 129, 130, 136, 153, 164, 205, 212, 221, 252, 255])
@pytest.mark.parametrize("axis", [1, 2])
def test_half_tile_columns(qsm, oracle, n, axis):
    rng = np.random.default_rng(n * 2 + axis)
    dims = [34, 6, 6]  # 17 half-spectrum columns: the last tile holds one
    dims[axis] = n
    dims = tuple(dims)
    size, vs, b = int(np.prod(dims)), (0.9, 1.1, 1.3), (0.2, -0.1, 1.0)
    chi = rng.standard_normal(size)
    f = qsm.dipole_forward(chi, qsm.Grid(dims, vs), b)
    # the bound of the dense-axis test: six FP32 transforms, each below 4e-7 of
    # its largest output
    assert np.max(np.abs(f - oracle.dipole_forward(chi, dims, vs, b))) < 6 * 4e-7 * np.max(np.abs(chi)) * 2
    field = rng.standard_normal(size) * 0.01
    m = (rng.random(size) < 0.8).astype(np.uint8)
    x = qsm.tv_admm(field, m, qsm.Grid(dims, vs), b, qsm.TvParams(lambda_=1e-3, rho=0.1, tol=0.0, max_iter=5))
    xo = oracle.tv_admm(field, m, dims, vs, b, 1e-3, 0.1, 0.0, 5)
    assert nrmse_dc(x, xo, m) < 2e-5  # FP32 against f64 on small volumes
