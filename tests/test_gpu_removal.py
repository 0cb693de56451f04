"""GPU tests of the removal planner and of the places of a captured run's
search phases: removals spread over few and many blocks, long neighbour
lists, foams at the size where the corrector stops forming its own sums, and
runs whose searches come after a different number of attempts."""
import numpy as np
import pytest

import cubble_amd as ca
from parity import FP64_TOL, assert_same_structure, attempt_errors, config, oracle_from_sim

pytestmark = pytest.mark.gpu

GAS = ca.IntegrationParams(True, False, True)


def _check_step(ora, sim, killed):
    """One accepted step with a removal, against the oracle from the same
    state; the pair count is that of the lists."""
    f = oracle_from_sim(ora, sim)
    before = sim.scalars()
    res = sim.integrate(GAS)
    f.integrate(True, True)
    gst, gsc = sim.get_state()
    ost, osc = f.get_state()
    assert gsc["count"] == osc["count"] == before["count"] - killed
    assert res["removals"] == before["removals"] + 1
    assert_same_structure(gst, ost)
    assert gsc["num_pairs"] == len(gst["nbr"]) // 2
    assert np.array_equal(gst["deg"], ost["deg"])
    assert np.allclose(gst["x"], ost["x"], rtol=1e-13, atol=1e-13)
    for key in ("vo", "saved"):
        assert np.array_equal(gst[key], ost[key]), key


# one deletion in each of `blocks` blocks of 256 bubbles (the planner sorts up
# to 1024 blocks, and walks them all beyond that), then two blocks' worth
@pytest.mark.parametrize("blocks", [1, 2, 63, 65, 1024, 1025])
def test_removal_spread_over_blocks(ora, blocks):
    print(f"removal over {blocks} blocks", flush=True)
    n = 270000
    sim = ca.Simulator(config(2, n, seed=50 + blocks))
    st, sc = sim.get_state()
    at = 256 * np.arange(blocks) + (np.arange(blocks) * 37) % 256
    st["x"][3][at] = 0.04
    sim.set_state(st, sc)
    _check_step(ora, sim, blocks)
    sim.close()


@pytest.mark.parametrize("dim,ipt", [(2, 1), (3, 1), (3, 4)])
def test_removal_filters_long_lists(ora, dim, ipt):
    """A bubble with more than 64 neighbours, some deleted and some moved from
    the tail (its list is rebuilt entry by entry), among ordinary ones."""
    print(f"long lists dim={dim} ipt={ipt}", flush=True)
    n = 4000
    sim = ca.Simulator(config(dim, n, seed=60 + dim),
                       tuning={"bubbles_per_thread": ipt, "search_tile": 64, "graph_steps": 8})
    st, sc = sim.get_state()
    st["x"][3][n // 2] = 9.0 if dim == 2 else 5.0
    sc["max_r_cell"] = float(st["x"][3].max())
    sim.set_state(st, sc)
    sim.search_neighbors()
    st, sc = sim.get_state()
    big = int(np.argmax(st["x"][3]))
    nb = st["nbr"][st["nbr_off"][big]:st["nbr_off"][big + 1]]
    assert len(nb) > 64
    kill = np.unique(np.concatenate([nb[::5], np.arange(0, n // 2, 29)]))
    kill = kill[kill != big]
    st["x"][3][kill] = 0.04
    sim.set_state(st, sc)
    _check_step(ora, sim, len(kill))
    sim.close()


# 255 to 257 blocks of 256 bubbles, around 128 and around 64 and 640 of them: the
# corrector forms the sums by waves, by workgroups, or leaves them to a launch
@pytest.mark.parametrize("n", [65, 16384, 16385, 32767, 32768, 32769, 65279, 65536, 65537,
                               163840, 163841])
def test_attempt_around_the_fused_sums(ora, n):
    print(f"fused sums n={n}", flush=True)
    sim = ca.Simulator(config(2, n, seed=70))
    f = oracle_from_sim(ora, sim)
    sim.step(GAS)
    f.attempt(True, True)
    sc = sim.scalars()
    errs = attempt_errors(2, sim.get_attempt(), f.attempt_out(), sc["f0"])
    for q, e in errs.items():
        assert e <= FP64_TOL, (q, e)
    osc = f.get_state()[1]
    for k in ("s_a", "s_ar", "s_oa", "s_oar"):
        assert sc[k] == pytest.approx(osc[k], rel=1e-11)
    sim.close()


@pytest.mark.parametrize("dim,n,precision", [(2, 900, ca.PREC_FP64), (3, 5000, ca.PREC_MIXED)])
def test_search_phase_places_do_not_change_a_run(dim, n, precision):
    """Foams wait for their search until the phase that ends a graph or comes
    every few attempts: runs with graphs of 1, 5 and 16 attempts, and one step
    per call, agree bit for bit."""
    print(f"search phases dim={dim} n={n}", flush=True)
    cfg = config(dim, n, seed=80, precision=precision, kappa=0.1)
    ends = []
    for groups in (1, 5, 16, 0):
        sim = ca.Simulator(cfg, tuning={"graph_steps": groups} if groups else None)
        if groups:
            res = sim.run_steps(300, GAS)
        else:
            for _ in range(300):
                res = sim.integrate(GAS)
        ends.append((sim.get_state()[0], res))
        sim.close()
    for st, res in ends[1:]:
        assert res == ends[0][1]
        for key in st:
            assert np.array_equal(st[key], ends[0][0][key]), key
    assert ends[0][1]["searches"] >= 3


@pytest.mark.parametrize("precision", [ca.PREC_FP64, ca.PREC_MIXED])
def test_removals_by_the_predictor_or_a_launch(precision):
    """A removal is carried out by the next attempt's predictor (captured runs
    of up to 2048 blocks), by a launch before the search phase, or by a launch
    after every attempt (larger runs, and one step per call): the same foams
    come out bit for bit."""
    print(f"removal routes precision={precision}", flush=True)
    small = [config(2, 3001, seed=91, precision=precision, kappa=1.0, r_std=0.3),
             config(3, 9000, seed=92, precision=precision, kappa=1.0, r_std=0.3)]
    large = config(2, 2048 * 256 + 1, seed=93, precision=precision)
    ends = []
    for cfgs, groups, calls in ((small, 16, False), (small, 3, False), (small, 0, True),
                                (small + [large], 16, False)):
        batch = ca.Batch(cfgs, tuning={"graph_steps": groups} if groups else None)
        if calls:
            for _ in range(400):
                res = batch.integrate(GAS)
        else:
            res = batch.run_steps(400, GAS)
        ends.append([(batch.get_state(k)[0], res[k]) for k in range(2)])
        batch.close()
    for end in ends[1:]:
        for (st, res), (st0, res0) in zip(end, ends[0]):
            assert res == res0
            for key in st:
                assert np.array_equal(st[key], st0[key]), key
    assert all(res["removals"] >= 20 for _, res in ends[0])
