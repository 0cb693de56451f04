"""GPU tests of remove_bubbles where the deletion marks are not those of the
state it finds: carried out already, of another count, of another launch shape.
Marks without a removal to carry out change nothing."""
import numpy as np
import pytest

import cubble_amd as ca
from parity import assert_same_structure, config, oracle_from_sim

pytestmark = pytest.mark.gpu

GAS = ca.IntegrationParams(True, False, True)


def _unchanged_by_removal(sim):
    st, sc = sim.get_state()
    sim.remove_bubbles()
    st1, sc1 = sim.get_state()
    assert sc1 == sc
    for key in st:
        assert np.array_equal(st1[key], st[key]), key


def _foam(dim, n, kill, seed=7):
    sim = ca.Simulator(config(dim, n, seed=seed))
    st, sc = sim.get_state()
    st["x"][3][kill] = 0.04
    sim.set_state(st, sc)
    return sim


# the last bubble, some at the end and some before, and more than a workgroup
@pytest.mark.parametrize("dim,n,kill", [(2, 3000, [2999]), (3, 2000, [5, 1000, 1997, 1998, 1999]),
                                        (2, 5000, list(range(4000, 5000, 2)))])
def test_marks_that_integrate_carried_out(dim, n, kill):
    print(f"marks after integrate dim={dim} kill={len(kill)}", flush=True)
    sim = _foam(dim, n, kill)
    res = sim.integrate(GAS)
    assert res["removals"] == 1 and res["count"] == n - len(kill)
    for _ in range(2):
        _unchanged_by_removal(sim)
    sim.run_steps(20, GAS)
    sim.close()


def test_marks_used_once():
    n = 3000
    kill = list(range(0, n, 31)) + [n - 1]
    sim = _foam(3, n, kill)
    _unchanged_by_removal(sim)  # no attempt yet
    sim.step(GAS)
    sim.remove_bubbles()
    assert sim.scalars()["count"] == n - len(kill)
    _unchanged_by_removal(sim)
    sim.close()


def test_marks_of_another_count():
    n = 2500
    sim = _foam(2, n, [n - 3, n - 2, n - 1])
    sim.step(GAS)
    small = ca.Simulator(config(2, n - 5, seed=9))
    st, sc = small.get_state()
    small.close()
    sim.set_state(st, sc)
    _unchanged_by_removal(sim)
    sim.close()


@pytest.mark.parametrize("dim,n", [(2, 6000), (3, 4000)])
def test_marks_and_another_launch_shape(ora, dim, n):
    """The blocks' partition changes between the attempt and its removal."""
    print(f"marks and launch shape dim={dim}", flush=True)
    kill = list(range(3, n, 257)) + [n - 1]
    sim = _foam(dim, n, kill)
    f = oracle_from_sim(ora, sim)
    sim.step(GAS)
    f.attempt(True, True)
    sim.retune({"bubbles_per_thread": 4, "search_tile": 64, "graph_steps": 8})
    sim.remove_bubbles()
    f.remove()
    gst, gsc = sim.get_state()
    ost, osc = f.get_state()
    assert gsc["count"] == osc["count"] == n - len(kill)
    assert_same_structure(gst, ost)
    assert np.allclose(gst["x"][3], ost["x"][3], rtol=1e-14, atol=0)
    sim.close()
