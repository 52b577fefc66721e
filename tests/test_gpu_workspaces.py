"""Workspaces kept between calls and staged host copies: the same results on
reused (dirty) blocks, from several threads at once, around the staging chunk
size, and after the kept memory is given back."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(dims, seed):
    rng = np.random.default_rng(seed)
    n = int(np.prod(dims))
    return rng.standard_normal(n) * 0.01, (rng.random(n) < 0.8).astype(np.uint8)


def _call(qsm, dims, seed):
    f, m = _case(dims, seed)
    g, b = qsm.Grid(dims, (1.0, 0.9, 1.1)), (0.1, 0.0, 1.0)
    return (qsm.tkd(f, m, g, b), qsm.tv_admm(f, m, g, b, qsm.TvParams(1e-3, 0.1, 0.0, 4)),
            *qsm.vsharp_with_radii(f, m, g, [3.0, 2.0], 0.05))


def test_same_results_on_reused_blocks(qsm):
    # the second round runs on the first's blocks, of larger and smaller volumes
    shapes = [(48, 40, 32), (20, 18, 16), (50, 41, 30)]
    first = [_call(qsm, d, i) for i, d in enumerate(shapes)]
    second = [_call(qsm, d, i) for i, d in reversed(list(enumerate(shapes)))][::-1]
    qsm.release_cached_memory()
    third = [_call(qsm, d, i) for i, d in enumerate(shapes)]
    for a, b, c in zip(first, second, third):
        for x, y, z in zip(a, b, c):
            assert np.array_equal(x, y) and np.array_equal(x, z)


def test_threads(qsm):
    shapes = [(48, 40, 32), (36, 30, 28), (64, 20, 24), (33, 35, 31)]
    want = [_call(qsm, d, i) for i, d in enumerate(shapes)]
    got = [None] * len(shapes)

    def work(i):
        for _ in range(3):
            got[i] = _call(qsm, shapes[i], i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(shapes))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for a, b in zip(want, got):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))


# 2 MiB chunks of f64 are 262144 values: below, at, above, and several with a remainder
@pytest.mark.parametrize("dims", [(64, 64, 63), (64, 64, 64), (64, 64, 65), (128, 96, 107)])
def test_copies_around_chunk_size(qsm, oracle, dims):
    f, m = _case(dims, 3)
    vs, b = (1.0, 1.0, 1.0), (0.0, 0.0, 1.0)
    x = qsm.tkd(f, m, qsm.Grid(dims, vs), b)
    ref = oracle.tkd(f, m, dims, vs, b, 0.15)
    # FP32 transforms, multiplier at most 1 / 0.15
    assert np.max(np.abs(x - ref)) < 2e-6 / 0.15 * np.max(np.abs(f)) * 4
    assert np.all(x[m == 0] == 0.0)
