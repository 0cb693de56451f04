"""GPU tests of the neighbour-list kernel where its matrix tiles can go wrong:
counts around the tile sizes, workgroups of one and several tiles, pairs at
the cutoff to the last bits (decided in FP64), cells so crowded that a tile's
candidates take several passes, and bubbles outside a walled box.  Lists are
bit-exact against the oracle's search and, where small, its brute force."""
import numpy as np
import pytest

import cubble_amd as ca
from parity import assert_same_structure, config, oracle_from_sim

pytestmark = pytest.mark.gpu


def _search_equals_oracle(ora, sim, st, sc, brute=True):
    sim.set_state(st, sc)
    f = oracle_from_sim(ora, sim)
    sim.search_neighbors()
    f.search()
    gst, gsc = sim.get_state()
    ost, osc = f.get_state()
    assert_same_structure(gst, ost)
    assert np.array_equal(gst["x"], ost["x"])
    assert gsc["num_pairs"] == osc["num_pairs"] == len(gst["nbr"]) // 2
    if brute:
        assert np.array_equal(ca.half_pairs(gst["nbr_off"], gst["nbr"]), f.brute_pairs())
    return gst, gsc


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [31, 32, 33, 63, 64, 65, 1500, 2049])
@pytest.mark.parametrize("tile", [32, 64, 256])
def test_counts_around_the_tiles(ora, dim, n, tile):
    print(f"search tiles dim={dim} n={n} tile={tile}", flush=True)
    # sparse enough for five cells per axis at the smallest counts
    sim = ca.Simulator(config(dim, n, phi=0.3 if n < 100 else None, seed=n),
                       tuning={"search_tile": tile})
    st, sc = sim.get_state()
    rng = np.random.default_rng(n)
    st["x"][:dim] += rng.normal(0.0, 0.3, size=(dim, n))
    _search_equals_oracle(ora, sim, st, sc)
    sim.close()


@pytest.mark.parametrize("dim,wall", [(2, (0, 0, 0)), (2, (1, 0, 0)), (3, (0, 0, 0)),
                                      (3, (0, 1, 1))])
def test_pairs_at_the_cutoff(ora, dim, wall):
    """400 pairs whose distance is the cutoff r_i + r_j + skin to within a few
    units in the last place, or 1e-9 .. 1e-5 off it."""
    print(f"search cutoff dim={dim} wall={wall}", flush=True)
    n = 4000
    sim = ca.Simulator(config(dim, n, seed=11 + dim, wall=wall))
    st, sc = sim.get_state()
    rng = np.random.default_rng(dim)
    x = st["x"]
    a = rng.permutation(n)[:800].reshape(2, 400)
    u = rng.normal(size=(dim, 400))
    u /= np.linalg.norm(u, axis=0)
    cut = x[3][a[0]] + x[3][a[1]] + sc["skin"]
    off = np.where(rng.random(400) < 0.5, rng.integers(-3, 4, 400) * 2.0 ** -52,
                   10.0 ** rng.uniform(-9, -5, 400) * rng.choice([-1, 1], 400))
    x[:dim, a[1]] = x[:dim, a[0]] + u * cut * (1.0 + off)
    for k in range(dim):
        lo, hi = sc["lbb"][k], sc["tfr"][k]
        if wall[k]:
            x[k] = np.clip(x[k], lo, hi)
    _search_equals_oracle(ora, sim, st, sc)
    sim.close()


@pytest.mark.parametrize("dim,n,big", [(2, 6000, 12.0), (3, 12000, 3.2)])
@pytest.mark.parametrize("tile", [32, 256])
def test_crowded_cells(ora, dim, n, big, tile):
    """A large bubble makes cells of hundreds of bubbles, so a tile has more
    candidates than one pass holds."""
    print(f"search crowded dim={dim} n={n} tile={tile}", flush=True)
    sim = ca.Simulator(config(dim, n, seed=21 + dim), tuning={"search_tile": tile})
    st, sc = sim.get_state()
    st["x"][3][n // 3] = big
    sc["max_r_cell"] = float(st["x"][3].max())
    gst, gsc = _search_equals_oracle(ora, sim, st, sc, brute=False)
    assert min(gsc["cell_dim"][:dim]) >= 5
    assert n / np.prod(gsc["cell_dim"]) > (100 if dim == 2 else 60)
    sim.close()


@pytest.mark.parametrize("dim,wall", [(2, (1, 1, 0)), (3, (1, 1, 1)), (3, (1, 0, 0))])
@pytest.mark.parametrize("reach", [9.0, 1e7])
def test_bubbles_outside_a_walled_box(ora, dim, wall, reach):
    """Bubbles pushed past a wall stay in the edge cell, outside the window
    the matrix product's bound covers (and, far away, the range of its
    factors)."""
    print(f"search outside dim={dim} wall={wall}", flush=True)
    n = 3000
    sim = ca.Simulator(config(dim, n, seed=31 + dim, wall=wall))
    st, sc = sim.get_state()
    rng = np.random.default_rng(dim)
    out = rng.permutation(n)[:60]
    st["x"][0][out[:30]] = -rng.uniform(0.0, reach, 30)
    st["x"][0][out[30:]] = sc["tfr"][0] + rng.uniform(0.0, reach, 30)
    _search_equals_oracle(ora, sim, st, sc)
    sim.close()


@pytest.mark.parametrize("dim,wall", [(2, (0, 0, 0)), (2, (0, 1, 0)), (3, (0, 0, 0)),
                                      (3, (0, 0, 1))])
@pytest.mark.parametrize("n", [1500, 6000])
def test_bubbles_more_than_a_period_outside(ora, dim, wall, n):
    """One wrap leaves them outside, in an edge cell, so that under the minimum
    image they touch bubbles of cells that are not that one's neighbours: the
    cells decide which pairs may meet."""
    print(f"search off the period dim={dim} wall={wall} n={n}", flush=True)
    sim = ca.Simulator(config(dim, n, seed=41 + dim, wall=wall))
    st, sc = sim.get_state()
    rng = np.random.default_rng(n)
    far = rng.permutation(n)[:150].reshape(3, 50)
    L = [sc["interval"][k] for k in range(3)]
    for k in range(dim):
        if wall[k]:
            continue
        st["x"][k][far[0]] = -rng.uniform(1.0, 1.9, 50) * L[k]
        st["x"][k][far[1]] = rng.uniform(2.0, 2.9, 50) * L[k]
    st["x"][0][far[2]] = rng.uniform(2.0, 2.9, 50) * L[0]
    for _ in range(2):  # the second search finds most of them a period nearer
        gst, gsc = _search_equals_oracle(ora, sim, st, sc, brute=False)
        assert min(gsc["cell_dim"][k] for k in range(dim)) >= 5
        pairs = set(map(tuple, np.stack([np.repeat(np.arange(n), np.diff(gst["nbr_off"])),
                                         gst["nbr"]], 1).tolist()))
        assert all((j, i) in pairs for i, j in pairs)
        st, sc = gst, gsc
    sim.run_steps(5, ca.IntegrationParams(True, False, True))
    sim.close()
