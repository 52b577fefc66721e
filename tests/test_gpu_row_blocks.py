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


# the unrolled solver's rows follow the volume alone (its sum over blocks gives
# the gradient of lambda); blocks that fill a small part of their tile, and all of it.
# The problem and the bars against the oracle are those of test_gpu_adjoint.py
@pytest.mark.parametrize("nx", [20, 82, 143, 338])
def test_unrolled_batch_of_one_length_equals_single(qsm, oracle, nx):
    dims, nv = (nx, 13, 10), 3
    n = int(np.prod(dims))
    rng = np.random.default_rng(nx)
    f, chi_true = rng.standard_normal((nv, n)) * 0.02, rng.standard_normal((nv, n)) * 0.01
    m = (rng.random((nv, n)) < 0.85).astype(np.uint8)
    vs, b, lam0, rho, K = (1.0, 1.0, 1.0), (0.1, -0.2, 1.0), 2e-3, 0.1, 5
    cb = np.stack([2.0 * (oracle.tv_admm(f[v], m[v], dims, vs, b, lam0, rho, 0.0, K) - chi_true[v])
                   for v in range(nv)])
    g, p = qsm.Grid(dims, vs), qsm.TvParams(lambda_=lam0, rho=rho, tol=0.0, max_iter=K)
    df, dm, dc = (qsm.DeviceArray.from_numpy(a.ravel()) for a in (f, m, cb))
    dx, dg = qsm.DeviceArray(nv * n, np.float64), qsm.DeviceArray(nv * n, np.float64)
    u = qsm.TvUnrolled([(g, b, df.ptr + 8 * n * v, dm.ptr + n * v, dx.ptr + 8 * n * v) for v in range(nv)], p)
    u.forward()
    lam = u.backward([dc.ptr + 8 * n * v for v in range(nv)], [dg.ptr + 8 * n * v for v in range(nv)])
    u.close()
    chi, grad = dx.numpy().reshape(nv, n), dg.numpy().reshape(nv, n)
    for v in range(nv):
        one = qsm.tv_unrolled_vjp(f[v], m[v], g, b, p, cb[v])
        assert np.array_equal(one[0], chi[v]) and np.array_equal(one[1], grad[v]) and one[2] == lam[v]
        xo, go, lo = oracle.tv_unrolled_vjp(f[v], m[v], dims, vs, b, lam0, rho, K, cb[v])
        assert oracle.nrmse(chi[v], xo, m[v]) <= 2e-5
        assert np.linalg.norm(grad[v] - go) <= 2e-3 * np.linalg.norm(go)
        assert abs(lam[v] - lo) <= 5e-3 * abs(lo)
    for d in (df, dm, dc, dx, dg):
        d.free()
