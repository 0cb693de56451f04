"""The pair kernel that gives a bubble four lanes (small launches with one
bubble a thread) against the one that gives it one: the same sums in the same
order, so the velocities and overlaps are equal bit for bit."""
import numpy as np
import pytest

import cubble_amd as ca
from parity import config

pytestmark = pytest.mark.gpu


def _attempt(cfg, ipt, ip, big=0.0):
    # two bubbles a thread: the kernel with one lane a bubble
    sim = ca.Simulator(cfg, tuning={"bubbles_per_thread": ipt, "graph_steps": 8})
    for _ in range(3):
        sim.integrate(ip)
    st, sc = sim.get_state()
    if big:
        st["x"][3][len(st["x"][3]) // 2] = big
        sc["max_r_cell"] = max(sc["max_r_cell"], big)
    return sim, st, sc


def _outputs(sim, st, sc, ip):
    sim.set_state(st, sc)
    sim.search_neighbors()
    sim.step(ip)
    return sim.get_attempt(), sim.scalars()


# around the 64 bubbles of a workgroup and the 256 of a block, lists of more
# than 8 and (a large bubble) more than 64 entries, gas exchange off, flow and
# walls
@pytest.mark.parametrize("precision", [ca.PREC_FP64, ca.PREC_MIXED])
@pytest.mark.parametrize("dim,n,gas,flow,walls,big", [
    (2, 5, True, False, False, 0.0), (2, 63, True, False, False, 0.0),
    (3, 64, True, False, False, 0.0), (2, 65, False, False, True, 0.0),
    (3, 257, True, False, True, 0.0), (2, 3001, True, True, True, 0.0),
    (3, 3000, True, True, False, 0.0), (3, 5000, False, False, False, 0.0),
    (2, 4000, True, False, False, 9.0), (3, 4000, True, True, False, 5.0)])
def test_four_lanes_a_bubble(precision, dim, n, gas, flow, walls, big):
    print(f"pair quad precision={precision} dim={dim} n={n} gas={gas} flow={flow} walls={walls} big={big}", flush=True)
    over = {"wall": (0, 1, 0)} if walls else {}
    if flow:
        over.update(flow=1, flow_vel=(0.01, 0.0, 0.0), flow_lbb=(0.0, 0.3, 0.0),
                    flow_tfr=(0.4, 0.7, 1.0))
    cfg = config(dim, n, seed=100 + n, precision=precision, **over)
    ip = ca.IntegrationParams(gas, flow, True)
    one, st, sc = _attempt(cfg, 1, ip, big)
    two, _, _ = _attempt(cfg, 2, ip)
    (a, sa), (b, sb) = _outputs(one, st, sc, ip), _outputs(two, st, sc, ip)
    assert np.array_equal(a["vp"][:3], b["vp"][:3])
    assert np.array_equal(a["ov"], b["ov"])
    for k in ("s_a", "s_ar", "s_oa", "s_oar"):
        # the blocks' sums in another order: n roundings at most
        assert sa[k] == pytest.approx(sb[k], rel=n * 2.0 ** -52, abs=1e-300)
    if big:
        lists, _ = one.get_state()
        assert np.max(np.diff(lists["nbr_off"])) > 64
    one.close()
    two.close()


@pytest.mark.parametrize("precision", [ca.PREC_FP64, ca.PREC_MIXED])
def test_several_foams_in_a_small_launch(precision):
    """A foam's run does not depend on the foams beside it: each alone, and the
    three in one launch of few blocks and of many."""
    cfgs = [config(d, n, seed=s, precision=precision)
            for d, n, s in ((2, 700, 7), (3, 1500, 8), (2, 300, 9))]
    large = config(3, 1024 * 256 + 1, seed=10, precision=precision)
    ip = ca.IntegrationParams()
    alone = []
    for c in cfgs:
        sim = ca.Simulator(c)
        sim.run_steps(40, ip)
        alone.append(sim.get_state()[0])
        sim.close()
    for group in (cfgs, cfgs + [large]):
        batch = ca.Batch(group)
        batch.run_steps(40, ip)
        for k, st in enumerate(alone):
            got = batch.get_state(k)[0]
            for key in st:
                assert np.array_equal(got[key], st[key]), (k, key)
        batch.close()
