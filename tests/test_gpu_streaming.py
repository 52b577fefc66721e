"""The non-temporal forms of the TV iteration's passes, which a batch larger
than the Infinity Cache runs: the same arithmetic, so the same bits as the
ordinary forms that each of its volumes runs alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [
    # compiled rows above and below 256, two-stage and staged z, the last
    # block partly empty; run-time rows of one, two and four columns a lane
    [(256, 205, 64), (320, 61, 96), (192, 192, 167)],
    [(164, 205, 131), (62, 300, 190), (125, 331, 64), (254, 129, 15)],
])
def test_batch_equals_alone(qsm, shapes):
    rng = np.random.default_rng(3)
    params = qsm.TvParams(lambda_=1e-3, rho=0.1, tol=1e-300, max_iter=4)
    vols, keep, outs = [], [], []
    # enough copies of the shapes that the batch is large whatever it counts
    copies = -(-(500 << 20) // (40 * sum(int(np.prod(s)) for s in shapes)))
    for dims in shapes * copies:
        n = int(np.prod(dims))
        f = qsm.DeviceArray.from_numpy(rng.standard_normal(n) * 0.01)
        m = qsm.DeviceArray.from_numpy((rng.random(n) < 0.8).astype(np.uint8))
        chi = qsm.DeviceArray(n, np.float64)
        keep.append((f, m))
        outs.append(chi)
        vols.append((qsm.Grid(dims, (1.0, 0.9, 1.1)), (0.1, 0.0, 1.0), f.ptr, m.ptr, chi.ptr))
    batch = qsm.TvBatch(vols, params)
    batch.run()
    together = [(batch.status(v), outs[v].numpy()) for v in range(len(vols))]
    batch.close()
    for v, vol in enumerate(vols):
        one = qsm.TvBatch([vol], params)
        one.run()
        assert one.status(0) == together[v][0]
        assert np.array_equal(outs[v].numpy(), together[v][1]), shapes[v % len(shapes)]
        one.close()
