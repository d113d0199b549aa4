"""Training on the device: the sample order is the sequential shuffle's, and the
target statistics and a whole small training agree with the same steps in
numpy."""
import numpy as np
import pytest

import tess

pytestmark = pytest.mark.gpu

M64 = (1 << 64) - 1


def _splitmix(state):
    state = (state + 0x9E3779B97F4A7C15) & M64
    z = state
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
    return state, z ^ (z >> 31)


def _fisher_yates(seed, epochs, n):
    state, orders = seed, []
    for _ in range(epochs):
        p = list(range(n))
        for i in range(n - 1, 0, -1):
            state, z = _splitmix(state)
            j = z % (i + 1)
            p[i], p[j] = p[j], p[i]
        orders.append(p)
    return orders


# one and several workgroups, one scan launch (up to 16,384) and three
@pytest.mark.parametrize("n", [1, 2, 3, 32, 255, 256, 257, 4097, 16384, 16385, 50000])
@pytest.mark.parametrize("seed", [0, 7, M64 - 3])
def test_shuffle_is_sequential(ctx, n, seed):
    for epoch, want in enumerate(_fisher_yates(seed, 2, n)):
        assert np.array_equal(ctx.diag_shuffle(seed, epoch, n), np.array(want, np.int32)), epoch


# rows at the edges of a workgroup's 256 and of all 65,536 threads.  The sums
# are in double, so the norm is the float nearest to the exact value or, where
# two are near, its neighbour: one unit in the last place.
@pytest.mark.parametrize("n", [255, 257, 3001, 66000])
def test_target_statistics(ctx, n):
    pts = tess.uniform(n, n)
    d = tess.Diagram(ctx, pts, np.zeros(3), np.ones(3), collect_stats=True)
    d.compute()
    st = d.stats()
    _, size, _ = d.grid()
    t = np.stack([np.log(np.sqrt(st["r2"]) / size.min()), np.log1p(st["classified"].astype(np.float64))], 1)
    m = tess.Model(ctx, seed=1)
    m.add_samples(d)
    m.train(epochs=1, batch=64, lr=1e-3, seed=3)
    norm = np.asarray(m.get()[1], np.float64)
    t = t.astype(np.float32).astype(np.float64)
    want = np.array([t[:, 0].mean(), t[:, 0].std(), t[:, 1].mean(), t[:, 1].std()])
    # the device's log may round a target the other way: one float unit of
    # 1.2e-7 in a few of n rows moves a mean or deviation by less than that
    assert np.allclose(norm, want, rtol=2.4e-7, atol=2.4e-7), (norm, want)
    m.close()
    d.close()
