"""GPU tests of removals of many bubbles at once, which foams of more than 256
blocks leave to launches of their own: against the oracle, the same foam run
and driven step by step, and the time of one."""
import time

import numpy as np
import pytest

import cubble_amd as ca
from parity import assert_same_structure, config, oracle_from_sim

pytestmark = pytest.mark.gpu

GAS = ca.IntegrationParams(True, False, True)


def _foam(dim, n, kill, tuning=None, precision=ca.PREC_FP64, seed=17):
    sim = ca.Simulator(config(dim, n, seed=seed, precision=precision), tuning=tuning)
    st, sc = sim.get_state()
    st["x"][3][kill] = 0.04
    sim.set_state(st, sc)
    return sim


def _kill(n, count, tail):
    rng = np.random.default_rng(n + count)
    head = rng.permutation(n - 2000)[:count - tail]
    return np.concatenate([head, np.arange(n - tail, n)])


# 256 and 257 deletions on both sides of 256 blocks; tails; half the foam
@pytest.mark.parametrize("n,count,tail", [(65536, 257, 3), (65537, 256, 3), (65537, 257, 3),
                                          (65537, 257, 257), (70000, 300, 0), (70000, 33000, 900)])
@pytest.mark.parametrize("dim,ipt", [(2, 1), (3, 2)])
def test_many_removed_in_one_step(ora, dim, ipt, n, count, tail):
    print(f"many removed dim={dim} n={n} count={count} ipt={ipt}", flush=True)
    kill = _kill(n, count, tail)
    sim = _foam(dim, n * ipt, kill, {"bubbles_per_thread": ipt, "search_tile": 64,
                                     "graph_steps": 8})
    f = oracle_from_sim(ora, sim)
    res = sim.integrate(GAS)
    f.integrate(True, True)
    gst, gsc = sim.get_state()
    ost, osc = f.get_state()
    assert res["count"] == gsc["count"] == osc["count"] == n * ipt - count
    assert res["removals"] == 1
    assert_same_structure(gst, ost)
    assert gsc["num_pairs"] == res["num_pairs"] == len(gst["nbr"]) // 2
    assert np.array_equal(gst["deg"], ost["deg"])
    assert np.allclose(gst["x"], ost["x"], rtol=1e-13, atol=1e-13)
    sim.close()


@pytest.mark.parametrize("precision", [ca.PREC_FP64, ca.PREC_MIXED])
def test_many_removed_in_a_run(precision):
    """In a captured run the foam waits for its plan; the others do not.  Runs
    with phases at different places and single steps agree bit for bit, in a
    foam alone and in batches on both sides of the predictor's removals."""
    print(f"many removed in a run precision={precision}", flush=True)
    n = 66000
    kill = _kill(n, 5000, 40)
    ends = []
    for groups in (16, 3, 0):
        sim = _foam(2, n, kill, {"graph_steps": groups} if groups else None, precision)
        if groups:
            res = sim.run_steps(40, GAS)
        else:
            for _ in range(40):
                res = sim.integrate(GAS)
        ends.append((sim.get_state()[0], res))
        sim.close()
    for st, res in ends[1:]:
        assert res == ends[0][1]
        for key in st:
            assert np.array_equal(st[key], ends[0][0][key]), key
    assert ends[0][1]["removals"] >= 1 and ends[0][1]["count"] <= n - 5000

    # bubbles that start at or below the smallest radius go together, one step
    # after the batch starts
    wide = [config(2, 66000, seed=4, precision=precision, r_std=0.5, r_lo=0.05, r_hi=1.5),
            config(2, 3000, seed=5, precision=precision, r_std=0.5, r_lo=0.05, r_hi=1.5)]
    large = config(2, 2048 * 256 + 1, seed=6, precision=precision)
    ends = []
    for cfgs, groups in ((wide, 16), (wide, 0), (wide + [large], 16)):
        batch = ca.Batch(cfgs, tuning={"graph_steps": groups} if groups else None)
        if groups:
            res = batch.run_steps(30, GAS)
        else:
            for _ in range(30):
                res = batch.integrate(GAS)
        ends.append([(batch.get_state(k)[0], res[k]) for k in range(2)])
        batch.close()
    for end in ends[1:]:
        for (st, res), (st0, res0) in zip(end, ends[0]):
            assert res == res0
            for key in st:
                assert np.array_equal(st[key], st0[key]), key
    assert ends[0][0][1]["removals"] >= 1 and ends[0][0][1]["count"] < 66000 - 256


def test_time_of_a_large_removal():
    """A removal is a small part of a step, not many steps' time: 20% of 3e5
    bubbles within 3 ms (planned by one workgroup 9)."""
    n = 300000
    kill = np.arange(0, n, 5)
    sim = _foam(3, n, kill)
    st, sc = sim.get_state()
    best = np.inf
    for _ in range(5):
        sim.set_state(st, sc)
        t = time.perf_counter()
        res = sim.integrate(GAS)
        best = min(best, time.perf_counter() - t)
        assert res["count"] <= n - len(kill)
    print(f"integrate with {len(kill)} removed: {best * 1e3:.2f} ms", flush=True)
    assert best < 3e-3
    sim.close()
