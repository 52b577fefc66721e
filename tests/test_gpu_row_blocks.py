"""Rows per block of run-time x lengths follow the launch: a volume gives the
same bits alone (2 to 8 rows a block here) and in a batch (6 to 16), whichever
rows a wave of the divergence fill takes one after the other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one, two and four columns a lane, register radices only; one, seven and eight
# rows of matrix tiles; two butterflies a row; rows of more than 256 columns
@pytest.mark.parametrize("nx", [20, 65, 82, 125, 143, 211, 251, 338])
def test_batch_of_one_length_equals_single(qsm, nx):
    dims, nv = (nx, 61, 40), 3
    n = int(np.prod(dims))
    rng = np.random.default_rng(nx)
    f, m = rng.standard_normal((nv, n)) * 0.01, (rng.random((nv, n)) < 0.8).astype(np.uint8)
    g, b = qsm.Grid(dims, (0.9, 1.0, 1.1)), (0.1, -0.2, 1.0)
    p, radii = qsm.TvParams(lambda_=1e-3, rho=0.1, tol=0.0, max_iter=5), [3.0, 2.0]
    df, dm = qsm.DeviceArray.from_numpy(f.ravel()), qsm.DeviceArray.from_numpy(m.ravel())
    dx, de = qsm.DeviceArray(nv * n, np.float64), qsm.DeviceArray(nv * n, np.uint8)
    at = lambda d, v, size: d.ptr + size * n * v
    tv = [(g, b, at(df, v, 8), at(dm, v, 1), at(dx, v, 8)) for v in range(nv)]
    vs = [(g, at(df, v, 8), at(dm, v, 1), at(dx, v, 8), at(de, v, 1)) for v in range(nv)]

    def run(make, vols):
        batch = make(vols)
        batch.run()
        batch.close()
        return dx.numpy().reshape(nv, n), de.numpy().reshape(nv, n)

    for make, vols in ((lambda v: qsm.TvBatch(v, p), tv), (lambda v: qsm.VsharpBatch(v, radii, 0.05), vs)):
        both, both_e = run(make, vols)
        for v in range(nv):
            one, one_e = run(make, vols[v:v + 1])
            assert np.array_equal(one[v], both[v]) and np.array_equal(one_e[v], both_e[v])
    for d in (df, dm, dx, de):
        d.free()
