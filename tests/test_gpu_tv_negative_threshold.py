"""Thresholds t = lambda / rho below 0 (the reference takes any), which run the
recording kernel in place of the clamped update, against the f64 oracle."""
import numpy as np
import pytest

from conftest import nrmse_dc


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(64, 9, 7), (200, 5, 8), (37, 11, 6), (129, 7, 9), (262, 6, 5), (352, 9, 7), (2, 3, 5)])
def test_tv_threshold_negative_against_oracle(qsm, oracle, dims):
    rng = np.random.default_rng(sum(dims))
    f = rng.standard_normal(int(np.prod(dims))) * 0.01
    m = (rng.random(f.size) < 0.8).astype(np.uint8)
    vs, b = (0.9, 1.0, 1.1), (0.1, -0.2, 1.0)
    x = qsm.tv_admm(f, m, qsm.Grid(dims, vs), b, qsm.TvParams(lambda_=-1e-3, rho=0.1, tol=0.0, max_iter=4))
    xo = oracle.tv_admm(f, m, dims, vs, b, -1e-3, 0.1, 0.0, 4)
    # the other TV tests' bound, or, where shrink's jump at v = t < 0 lies near
    # some value, what an FP32 rounding of the field alone does to the f64 result
    moved = oracle.tv_admm(f.astype(np.float32).astype(np.float64), m, dims, vs, b, -1e-3, 0.1, 0.0, 4)
    assert nrmse_dc(x, xo, m) < max(1e-5, 20 * nrmse_dc(moved, xo, m))
