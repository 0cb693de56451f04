"""One foam's integrate() works without step limits and reads its scalars with
the controller's launch: the same steps as a foam of a batch, whatever ran or
halted the foam before."""
import numpy as np
import pytest

import cubble_amd as ca
from parity import config

pytestmark = pytest.mark.gpu

IP = ca.IntegrationParams()


@pytest.mark.parametrize("dim,n,precision", [(2, 700, 0), (3, 1500, 1)])
def test_single_foam_steps_as_in_a_batch(dim, n, precision):
    cfg = config(dim, n, seed=5, precision=precision, kappa=0.5)
    batch = ca.Batch([cfg, config(2, 300, seed=6, precision=precision)])
    sim = ca.Simulator(cfg)
    for k in range(60):
        want = batch.integrate(IP)[0]
        assert sim.integrate(IP) == want, k
        if k == 20:
            sim.search_neighbors()  # (counted, and bubbles are reordered in both)
            sim.step(IP)
            st, sc = sim.get_state()
            break
    assert sc["steps"] == want["steps"] == 21
    batch.close()
    # the rest by one step a call and by one run
    other = ca.Simulator(cfg)
    other.set_state(st, sc)
    for _ in range(25):
        a = sim.integrate(IP)
    b = other.run_steps(25, IP)
    assert a == b
    got, want = sim.get_state()[0], other.get_state()[0]
    for key in got:
        assert np.array_equal(got[key], want[key]), key
    sim.close()
    other.close()


def test_a_stop_rule_halts_one_call_only():
    sim = ca.Simulator(config(2, 500, seed=7))
    sim.set_stop_rules(max_radius=1e-3)  # met by every step
    for k in range(1, 6):
        assert sim.integrate(IP)["steps"] == k
    assert sim.run_steps(3, IP)["steps"] >= 6
    steps = sim.scalars()["steps"]
    sim.set_stop_rules()
    sim.step(IP)
    assert sim.integrate(IP)["steps"] == steps + 1
    sim.close()
