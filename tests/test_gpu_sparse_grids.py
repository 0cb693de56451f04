"""GPU tests of boxes whose cell grid is cut down to the number of cells there
is room for: the grid is the documented one (one cell less on the axis with the
most, the first of equals, until they fit), lists and pairs are exact, and
finding it takes no time."""
import time

import numpy as np
import pytest

import cubble_amd as ca
from parity import assert_same_structure, config, oracle_from_sim
from test_gpu_pairs import brute, foam_positions, gpu_pairs

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dim,n,rel,factor,shrink", [
    (2, 3000, (1.0, 1.0, 1.0), 0.01, 1.0), (2, 3000, (5.0, 1.0, 1.0), 0.3, 0.3),
    (2, 3000, (1.0, 9.0, 1.0), 0.9, 0.1), (2, 3000, (1.0, 1.0, 1.0), 1.0, 0.01),
    (3, 3000, (1.0, 1.0, 1.0), 0.1, 1.0), (3, 3000, (3.0, 1.0, 2.0), 0.5, 0.3),
    (3, 3000, (1.0, 4.0, 4.0), 0.9, 0.1), (3, 3000, (7.0, 7.0, 1.0), 1.0, 0.01)])
def test_grid_cut_down_to_its_cells(ora, dim, n, rel, factor, shrink):
    print(f"sparse grid dim={dim} rel={rel} factor={factor} shrink={shrink}", flush=True)
    sim = ca.Simulator(config(dim, n, seed=3, rel_dim=rel, cell_cap_factor=factor))
    st, sc = sim.get_state()
    # smaller bubbles: more cells than the foam has room for
    st["x"][3] *= shrink
    sc["max_r_cell"] *= shrink
    sim.set_state(st, sc)
    f = oracle_from_sim(ora, sim)
    sim.search_neighbors()
    f.search()
    gst, gsc = sim.get_state()
    ost, osc = f.get_state()
    assert list(gsc["cell_dim"]) == list(osc["cell_dim"])
    assert np.prod(gsc["cell_dim"]) <= max(gsc["cell_cap"], 1)
    assert_same_structure(gst, ost)
    sim.close()


@pytest.mark.parametrize("dim,n,L", [(2, 3000, (1e5, 1e5, 0.0)), (3, 2000, (2e3, 9e3, 5e3))])
def test_pairs_of_a_sparse_box(ora, dim, n, L):
    print(f"sparse pairs dim={dim} L={L}", flush=True)
    x = foam_positions(np.random.default_rng(dim), dim, n, L)
    # neighbours for half of them
    h = n // 2
    x[:dim, h:] = x[:dim, :n - h] + np.random.default_rng(9).uniform(-1.5, 1.5, (dim, n - h))
    x[:dim] = np.clip(x[:dim], 0.0, np.array(L[:dim])[:, None])
    want = brute(ora, dim, L, (0, 0, 0), 0.3, x)
    assert len(want) > n // 4
    total, got = gpu_pairs(dim, L, (0, 0, 0), 0.3, x, 8 * n)
    assert total == len(want) and np.array_equal(got, want)


def test_time_of_a_sparse_box():
    """20,000 bubbles in a box a hundred thousand across, within 1 ms (every
    wave took the grid's cells down one by one: 44 ms)."""
    n, L = 20000, 1e5
    rng = np.random.default_rng(1)
    dev = [torch.tensor(rng.uniform(0.0, L, n), device="cuda") for _ in range(2)]
    r = torch.tensor(rng.uniform(0.5, 1.5, n), device="cuda")
    pi = torch.zeros(64, dtype=torch.int32, device="cuda")
    pj = torch.zeros_like(pi)
    num = torch.zeros(1, dtype=torch.int64, device="cuda")
    box = ca.Box.of(2, [0.0] * 3, [L, L, 0.0], (0, 0, 0))
    best = np.inf
    for _ in range(5):
        torch.cuda.synchronize()
        t = time.perf_counter()
        ca.find_pairs(dev[0].data_ptr(), dev[1].data_ptr(), 0, r.data_ptr(), n, box, 0.3,
                      pi.data_ptr(), pj.data_ptr(), 64, num.data_ptr(),
                      torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t)
    print(f"pairs of a sparse box: {best * 1e3:.2f} ms", flush=True)
    assert best < 1e-3
