"""GPU tests of removals that rebuild neighbour lists of thousands of entries
(a very large bubble among ordinary ones): against the oracle, and the time of
one."""
import time

import numpy as np
import pytest

import cubble_amd as ca
from parity import assert_same_structure, config, oracle_from_sim

pytestmark = pytest.mark.gpu

GAS = ca.IntegrationParams(True, False, True)


@pytest.mark.parametrize("frac,tail", [(0.0, 1), (0.02, 40), (0.3, 200), (0.9, 1500)])
@pytest.mark.parametrize("dim,n,big", [(2, 6000, 30.0), (3, 6000, 12.0)])
def test_lists_of_a_thousand(ora, dim, n, big, frac, tail):
    """A bubble with a list of about a thousand, which keeps, loses and renames few or
    most of its entries, in place and moved into a hole."""
    print(f"long lists dim={dim} frac={frac} tail={tail}", flush=True)
    sim = ca.Simulator(config(dim, n, seed=27 + dim))
    st, sc = sim.get_state()
    st["x"][3][[n // 3, n - 2]] = big  # the second one is a tail survivor
    sc["max_r_cell"] = big
    sim.set_state(st, sc)
    sim.search_neighbors()
    st, sc = sim.get_state()
    assert np.diff(st["nbr_off"]).max() > 800
    rng = np.random.default_rng(int(1000 * frac) + tail)
    kill = np.unique(np.concatenate([np.flatnonzero(rng.random(n) < frac),
                                     rng.permutation(n - 2000)[:tail]]))
    kill = kill[st["x"][3][kill] < big]
    st["x"][3][kill] = 0.04
    sim.set_state(st, sc)
    f = oracle_from_sim(ora, sim)
    sim.step(GAS)
    f.attempt(True, True)
    assert np.array_equal(sim.get_attempt()["del"], f.attempt_out()["del"])
    sim.remove_bubbles()
    f.remove()
    gst, gsc = sim.get_state()
    ost, osc = f.get_state()
    assert gsc["count"] == osc["count"] == n - len(kill)
    assert_same_structure(gst, ost)
    assert gsc["num_pairs"] == len(gst["nbr"]) // 2
    sim.close()


@pytest.mark.parametrize("keeps", [True, False])
def test_time_of_a_long_list(keeps):
    """Rebuilding a list of some thousand entries takes a wave a few hundred
    cycles per 64 of them, and so does marking what it names: a removal within
    0.5 ms (entry by entry 1.3)."""
    n = 20000
    sim = ca.Simulator(config(3, n, seed=37))
    st, sc = sim.get_state()
    st["x"][3][n // 2 + 1] = sc["max_r_cell"] = 18.0
    sim.set_state(st, sc)
    sim.search_neighbors()
    st, sc = sim.get_state()
    assert np.diff(st["nbr_off"]).max() > 4000
    small = np.arange(n) % 200 == (0 if keeps else np.argmax(st["x"][3]) % 200)
    st["x"][3][small] = 0.04
    best = np.inf
    for _ in range(4):
        sim.set_state(st, sc)
        sim.step(GAS)
        t = time.perf_counter()
        sim.remove_bubbles()
        best = min(best, time.perf_counter() - t)
        assert sim.scalars()["count"] < n
    print(f"removal with a list of thousands: {best * 1e3:.2f} ms", flush=True)
    assert best < 5e-4
    sim.close()
