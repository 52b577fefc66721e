"""The fused z/u update over the thresholds t = lambda / rho that the entry
points take, on compiled and run-time row lengths: t >= 0 (the clamped form)
against the f64 oracle (src/inversion/admm.rs:127-142, src/utils/mod.rs:
44-52), and t < 0, which runs the recording kernel, against the unrolled
solver that always does."""
import numpy as np
import pytest

from conftest import nrmse_dc


DIMS = [(64, 9, 7), (72, 10, 6), (200, 5, 8), (37, 11, 6), (63, 8, 5), (65, 3, 4), (125, 6, 7), (129, 7, 9), (253, 5, 6),
        (257, 4, 3), (262, 6, 5), (352, 9, 7), (505, 5, 4), (511, 6, 5), (1, 5, 4), (2, 3, 5)]


@pytest.mark.gpu
@pytest.mark.parametrize("lam", [1e-3, 0.0])
@pytest.mark.parametrize("dims", DIMS)
def test_tv_threshold_nonnegative(qsm, oracle, dims, lam):
    rng = np.random.default_rng(sum(dims))
    f = rng.standard_normal(int(np.prod(dims))) * 0.01
    m = (rng.random(f.size) < 0.8).astype(np.uint8)
    vs, b = (0.9, 1.0, 1.1), (0.1, -0.2, 1.0)
    # FP32 against f64 over 8 iterations: the other TV tests' bound
    x = qsm.tv_admm(f, m, qsm.Grid(dims, vs), b, qsm.TvParams(lambda_=lam, rho=0.1, tol=0.0, max_iter=8))
    xo = oracle.tv_admm(f, m, dims, vs, b, lam, 0.1, 0.0, 8)
    assert nrmse_dc(x, xo, m) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("dims", DIMS)
def test_tv_threshold_negative(qsm, dims):
    rng = np.random.default_rng(sum(dims))
    f = rng.standard_normal(int(np.prod(dims))) * 0.01
    m = (rng.random(f.size) < 0.8).astype(np.uint8)
    b = (0.1, -0.2, 1.0)
    p = qsm.TvParams(lambda_=-1e-3, rho=0.1, tol=0.0, max_iter=8)
    grid = qsm.Grid(dims, (0.9, 1.0, 1.1))
    x = qsm.tv_admm(f, m, grid, b, p)
    chi, _, _ = qsm.tv_unrolled_vjp(f, m, grid, b, p, np.zeros(f.size))
    assert np.array_equal(x, chi)
