"""Pixel distances where a call's distinct wavelengths come near the number that
are evaluated once each, and with the NaN that marks free table entries."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,distinct", [(4096, 3000), (4097, 3000), (8192, 3400), (20000, 4096), (20000, 4097),
                                        (20000, 4400), (20000, 12000), (100000, 3300), (100000, 60000)])
def test_distances_around_the_list_limit(dev, n, distinct):
    rng = np.random.default_rng(n + distinct)
    pool = np.unique(rng.uniform(3.3, 3.75, 3 * distinct).astype(np.float32))
    rng.shuffle(pool)
    pool = pool[:distinct]
    small = np.concatenate([dev.pixel_distances(pool[s:s + 300]) for s in range(0, distinct, 300)])
    pick = np.concatenate([np.arange(distinct), rng.integers(0, distinct, n)])[:n]
    rng.shuffle(pick)
    assert np.array_equal(dev.pixel_distances(pool[pick]), small[pick])


@pytest.mark.parametrize("n", [1, 700, 5000, 50000])
def test_the_nan_of_all_ones(dev, n):
    rng = np.random.default_rng(n)
    pool = np.unique(rng.uniform(3.3, 3.75, 900).astype(np.float32))
    x = pool[rng.integers(0, len(pool), n)]
    want = dev.pixel_distances(pool)[np.searchsorted(pool, x)]
    odd = rng.random(n) < 0.01
    odd[-1] = True
    y = x.copy()
    y.view(np.uint32)[odd] = 0xffffffff
    d = dev.pixel_distances(y)
    assert np.isnan(d[odd]).all() and np.array_equal(d[~odd], want[~odd])
