"""GPU tests of cubble_find_pairs where its matrix tiles and sorting can go
wrong: counts around the tile sizes, pairs at the cutoff to the last bits,
bubbles with more pairs than are sorted in LDS, bubbles outside the box (past
walls, and more than a period off), and grids of every kind -- against the
oracle's brute force or, for positions it does not wrap, a direct walk of the
documented rule."""
import numpy as np
import pytest

import cubble_amd as ca
from test_gpu_pairs import brute, foam_positions, gpu_pairs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 31, 33, 64, 65, 127, 1025, 4097])
def test_counts_around_the_tiles(ora, dim, n):
    print(f"pairs tiles dim={dim} n={n}", flush=True)
    rng = np.random.default_rng(n)
    # half of full density, at least six cells per axis
    edge = max((n * (3.0 if dim == 2 else 8.0)) ** (1.0 / dim), 6 * 3.5)
    L = (edge, edge * 1.3, edge * 0.9)
    x4 = foam_positions(rng, dim, n, L)
    want = brute(ora, dim, L, (0, 0, 0), 0.3, x4)
    for noalloc in (False, True):
        total, got = gpu_pairs(dim, L, (0, 0, 0), 0.3, x4, 64 * n,
                               lambda *a: ca.find_pairs(*a, noalloc=noalloc))
        assert total == len(want) and np.array_equal(got, want)


@pytest.mark.parametrize("dim,wall", [(2, (0, 0, 0)), (2, (0, 1, 0)), (3, (0, 0, 0)),
                                      (3, (1, 1, 0))])
def test_pairs_at_the_cutoff(ora, dim, wall):
    print(f"pairs cutoff dim={dim} wall={wall}", flush=True)
    n, skin = 4000, 0.3
    L = (110.0, 110.0, 0.0) if dim == 2 else (32.0, 27.0, 36.0)
    rng = np.random.default_rng(40 + dim)
    x = foam_positions(rng, dim, n, L)
    a = rng.permutation(n)[:800].reshape(2, 400)
    u = rng.normal(size=(dim, 400))
    u /= np.linalg.norm(u, axis=0)
    cut = x[3][a[0]] + x[3][a[1]] + skin
    off = np.where(rng.random(400) < 0.5, rng.integers(-3, 4, 400) * 2.0 ** -52,
                   10.0 ** rng.uniform(-9, -5, 400) * rng.choice([-1, 1], 400))
    x[:dim, a[1]] = x[:dim, a[0]] + u * cut * (1.0 + off)
    for k in range(dim):  # inside the box, where the oracle's brute force is defined
        x[k] = np.clip(x[k], 0.0, L[k]) if wall[k] else np.where(
            x[k] < 0, x[k] + L[k], np.where(x[k] > L[k], x[k] - L[k], x[k]))
    want = brute(ora, dim, L, wall, skin, x)
    total, got = gpu_pairs(dim, L, wall, skin, x, 64 * n)
    assert total == len(want) and np.array_equal(got, want)


@pytest.mark.parametrize("dim,n,r", [(2, 3000, 9.0), (3, 6000, 3.3)])
def test_bubbles_with_many_pairs(ora, dim, n, r):
    """Large bubbles with 33 and more larger-index neighbours, first in index
    order; with and without room for all pairs."""
    print(f"pairs many dim={dim}", flush=True)
    L = (100.0, 100.0, 0.0) if dim == 2 else (38.0, 38.0, 38.0)
    rng = np.random.default_rng(50 + dim)
    x = foam_positions(rng, dim, n, L)
    x[3][:5] = r
    want = brute(ora, dim, L, (0, 0, 0), 0.3, x)
    assert np.bincount(want[:, 0])[:5].min() > 32
    total, got = gpu_pairs(dim, L, (0, 0, 0), 0.3, x, 64 * n)
    assert total == len(want) and np.array_equal(got, want)
    whole, end = np.searchsorted(want[:, 0], [2, 3])
    cap = int(end) - 1  # cut inside bubble 2's group
    total, got = gpu_pairs(dim, L, (0, 0, 0), 0.3, x, cap)
    assert total == len(want)
    assert np.array_equal(got[:whole], want[:whole]) and np.all(got[whole:, 0] == 2)
    assert np.all(np.diff(got[whole:, 1]) > 0)
    assert set(got[whole:, 1]) <= set(want[want[:, 0] == 2][:, 1])


def _rule(dim, L, wall, skin, x4):
    """The documented result by direct tests: positions wrapped once, cells of
    edge at least 2 (max r + skin) by clamped index, pairs of neighbouring
    cells within reach under the minimum image."""
    n = x4.shape[1]
    p = np.zeros((3, n))
    for k in range(dim):
        v = x4[k]
        p[k] = v if wall[k] else np.where(v < 0, v + L[k], np.where(v > L[k], v - L[k], v))
    edge = 2 * (x4[3].max() + skin)
    cd = [max(1, int(np.floor(L[k] / edge))) if k < dim else 1 for k in range(3)]
    c = [np.clip(np.floor(cd[k] * p[k] / L[k]), 0, cd[k] - 1).astype(int) if k < dim
         else np.zeros(n, int) for k in range(3)]
    out = []
    for i in range(n):
        ok = np.arange(n) > i
        m = np.zeros(n)
        for k in range(dim):
            dc = np.abs(c[k] - c[k][i])
            ok &= (dc <= 1) if wall[k] else (np.minimum(dc, cd[k] - dc) <= 1)
            d = p[k][i] - p[k]
            t = L[k] - np.abs(d)
            image = np.where(d < 0, t, -t)
            d = d if wall[k] else np.where(t * t < d * d, image, d)
            m = m + d * d
        cut = x4[3][i] + x4[3] + skin
        out += [(i, j) for j in np.flatnonzero(ok & (m < cut * cut))]
    return np.array(out, dtype=np.int32).reshape(-1, 2)


@pytest.mark.parametrize("dim,wall", [(2, (0, 0, 0)), (2, (1, 0, 0)), (3, (0, 0, 0)),
                                      (3, (1, 1, 1)), (3, (0, 1, 0))])
def test_bubbles_outside_the_box(dim, wall):
    print(f"pairs outside dim={dim} wall={wall}", flush=True)
    n = 1500
    L = (60.0, 48.0, 0.0) if dim == 2 else (24.0, 20.0, 22.0)
    rng = np.random.default_rng(60 + dim)
    x = foam_positions(rng, dim, n, L)
    far = rng.permutation(n)[:150].reshape(3, 50)
    for k in range(dim):
        x[k, far[0]] -= rng.uniform(0.0, 1.0, 50) * L[k]          # up to a period below
        x[k, far[1]] += rng.uniform(0.9, 2.6, 50) * L[k]          # up to two and a half above
    x[0, far[2]] = -rng.uniform(1.0, 2.2, 50) * L[0]
    want = _rule(dim, L, wall, 0.3, x)
    total, got = gpu_pairs(dim, L, wall, 0.3, x, 64 * n)
    assert total == len(want) and np.array_equal(got, want)
