"""GPU tests of the matrix tiles' band: pairs whose |d|^2 is off the cutoff's
square by 0.3 to 10 times the bound within which the tiles leave a pair to FP64,
on both sides, for windows of 1 to 10 cells.  Narrower or wider, the lists are
those of the FP64 test."""
import numpy as np
import pytest

import cubble_amd as ca
from parity import assert_same_structure, config, oracle_from_sim
from test_gpu_pairs import brute, foam_positions, gpu_pairs

pytestmark = pytest.mark.gpu

BAND = 22 * 2.0 ** -22


def _band(dim, e, hr, kx):
    """The bound of |d|^2 - cutoff^2 for windows of kx cells of edges e."""
    h = [(0.5 * kx + 1.0) * e[0], 1.5 * e[1], 1.5 * e[2] if dim == 3 else np.zeros_like(kx)]
    return BAND * 1.001 * (h[0] ** 2 + h[1] ** 2 + h[2] ** 2 + hr * hr)


def _plant(rng, x, dim, skin, pairs, band):
    """Moves one bubble of each of `pairs` disjoint pairs to a distance whose
    square is off the cutoff's by 0.3 to 10 bands."""
    a = rng.permutation(x.shape[1])[:2 * pairs].reshape(2, pairs)
    u = rng.normal(size=(dim, pairs))
    u /= np.linalg.norm(u, axis=0)
    off = 10.0 ** rng.uniform(np.log10(0.3), 1.0, pairs) * rng.choice([-1, 1], pairs) * band
    cut = x[3][a[0]] + x[3][a[1]] + skin
    x[:dim, a[1]] = x[:dim, a[0]] + u * np.sqrt(cut ** 2 + off)


# ordinary cells (tiles of many), and cells widened by a large bubble (of few)
@pytest.mark.parametrize("dim,n,big", [(2, 12000, None), (2, 12000, 4.0), (2, 12000, 9.0),
                                       (3, 20000, None), (3, 20000, 2.2), (3, 20000, 3.0)])
def test_lists_at_the_band(ora, dim, n, big):
    print(f"band lists dim={dim} big={big}", flush=True)
    sim = ca.Simulator(config(dim, n, seed=51 + dim))
    for seed in range(3):
        st, sc = sim.get_state()
        rng = np.random.default_rng(seed)
        if big:
            st["x"][3][7] = big
        sc["max_r_cell"] = max_r = float(st["x"][3].max())
        skin = sc["skin"]
        cells = [max(1, int(sc["interval"][k] // (2 * (max_r + skin)))) for k in range(dim)]
        assert min(cells) >= 5
        e = [sc["interval"][k] / cells[k] for k in range(dim)]
        pairs = n // 3
        _plant(rng, st["x"], dim, skin, pairs,
               _band(dim, e, max_r + skin, rng.integers(1, 11, pairs).astype(float)))
        sim.set_state(st, sc)
        f = oracle_from_sim(ora, sim)
        sim.search_neighbors()
        f.search()
        gst, gsc = sim.get_state()
        assert list(gsc["cell_dim"][:dim]) == cells
        ost, _ = f.get_state()
        assert_same_structure(gst, ost)
    sim.close()


@pytest.mark.parametrize("dim,wall,big", [(2, (0, 0, 0), 1.4), (2, (0, 1, 0), 5.0),
                                          (3, (0, 0, 0), 1.4), (3, (1, 0, 0), 2.4)])
def test_pairs_at_the_band(ora, dim, wall, big):
    print(f"band pairs dim={dim} wall={wall} big={big}", flush=True)
    n, skin = 6000, 0.3
    L = (140.0, 130.0, 0.0) if dim == 2 else (40.0, 36.0, 44.0)
    for seed in range(3):
        rng = np.random.default_rng(60 + seed)
        x = foam_positions(rng, dim, n, L)
        x[3][5] = big
        max_r = x[3].max()
        cells = [int(L[k] // (2 * (max_r + skin))) for k in range(dim)]
        assert min(cells) >= 5
        e = [L[k] / cells[k] for k in range(dim)]
        pairs = n // 3
        kx = rng.integers(1, 11, pairs).astype(float)
        # two roundings more, and the positions' steps of 2^-32 of a box
        band = (26.0 / 22.0 * _band(dim, e, max_r + skin, kx) +
                16 * (2 * max_r + skin) * max(L) * 2.0 ** -31)
        _plant(rng, x, dim, skin, pairs, band)
        for k in range(dim):  # inside the box, where the oracle's brute force is defined
            x[k] = np.clip(x[k], 0.0, L[k]) if wall[k] else np.where(
                x[k] < 0, x[k] + L[k], np.where(x[k] > L[k], x[k] - L[k], x[k]))
        want = brute(ora, dim, L, wall, skin, x)
        total, got = gpu_pairs(dim, L, wall, skin, x, 64 * n)
        assert total == len(want) and np.array_equal(got, want)
