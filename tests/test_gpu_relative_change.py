"""The change an iteration reports (src/utils/mod.rs:69-77) where no iteration
can stop the run: with tol <= 0 only the last iteration forms it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(64, 12, 10),    # compiled rows, quarter-row blocks
                                  (256, 9, 5),     # compiled rows, an odd number of them
                                  (82, 7, 5),      # run-time rows
                                  (600, 5, 3)])    # run-time rows above 512
@pytest.mark.parametrize("iters", [1, 2, 3, 4, 9])
@pytest.mark.parametrize("graphs", [True, False])
def test_status_without_a_stop_test(qsm, dims, iters, graphs):
    # A tol no change falls below runs the same iterations and forms every
    # change: the same sums in the same order, so the same bits.
    rng = np.random.default_rng(5)
    n = int(np.prod(dims))
    f = qsm.DeviceArray.from_numpy(rng.standard_normal(n) * 0.01)
    m = qsm.DeviceArray.from_numpy((rng.random(n) < 0.8).astype(np.uint8))
    got = []
    for tol in (1e-300, 0.0, -1.0, float("nan")):
        chi = qsm.DeviceArray(n, np.float64)
        b = qsm.TvBatch([(qsm.Grid(dims, (1.0, 0.9, 1.1)), (0.1, 0.0, 1.0), f.ptr, m.ptr, chi.ptr)],
                        qsm.TvParams(lambda_=1e-3, rho=0.1, tol=tol, max_iter=iters))
        if not graphs:
            b.set_graphs(False)
        for _ in range(2):
            b.run()
            got.append((b.status(0), chi.numpy().tobytes()))
        b.close()
    assert got[0][0][0] == iters and got[0][0][1] > 0
    for g in got[1:]:
        assert g == got[0]
