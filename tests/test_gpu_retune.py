"""GPU test of new launch shapes for one foam: they take no block tables, so they
cost the same for a large foam as for a small one, and change no result."""
import time

import numpy as np
import pytest

import cubble_amd as ca
from parity import config

pytestmark = pytest.mark.gpu

GAS = ca.IntegrationParams(True, False, True)
SHAPES = [{"bubbles_per_thread": 0, "search_tile": t, "graph_steps": 0} for t in (0, 64)]


def _best(sim):
    best = np.inf
    for k in range(12):
        t = time.perf_counter()
        sim.retune(SHAPES[k % 2])
        best = min(best, time.perf_counter() - t)
    return best


def test_time_of_new_shapes():
    times = []
    for n in (1000, 4000000):
        sim = ca.Simulator(config(3, n, seed=2, precision=ca.PREC_MIXED))
        times.append(_best(sim))
        sim.close()
    print("retune: %.1f us, %.1f us" % tuple(1e6 * t for t in times), flush=True)
    assert times[1] < 3 * times[0]


def test_new_shapes_between_steps():
    ends = []
    for change in (False, True):
        sim = ca.Simulator(config(2, 5000, seed=2))
        for k in range(4):
            if change:
                sim.retune(SHAPES[k % 2])
            res = sim.run_steps(20, GAS)
        ends.append((sim.get_state()[0], res))
        sim.close()
    assert ends[0][1] == ends[1][1]
    for key in ends[0][0]:
        assert np.array_equal(ends[0][0][key], ends[1][0][key]), key
