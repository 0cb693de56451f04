"""Read-back of a foam's state in chunks through pinned memory: states written
from the host come back whole, whatever the chunks' borders cut, and from
several threads at once.  Nothing is computed, so the values are equal."""
import threading

import numpy as np
import pytest

import cubble_amd as ca

pytestmark = pytest.mark.gpu


def _state(n, dim, mixed, seed):
    rng = np.random.default_rng(seed)

    def narrow(a):  # what mixed precision holds in FP32
        return a.astype(np.float32).astype(np.float64) if mixed else a

    st = {k: rng.uniform(0.1, 0.9, (4, n)) for k in ("x", "v", "vo", "saved")}
    for k in ("v", "vo", "saved"):
        st[k] = narrow(st[k])
    if dim == 2:
        for k in ("x", "v", "vo", "saved"):
            st[k][2] = 0.0
    st["path"], st["err"] = rng.random(n), narrow(rng.random(n))
    st["wc"] = rng.integers(-5, 5, (3, n)).astype(np.int32)
    st["wc"][dim:] = 0
    st["idx"] = rng.permutation(n).astype(np.int32)
    st["deg"] = rng.integers(0, 9, n).astype(np.int32)
    # uneven symmetric lists, some empty
    a = np.arange(n, dtype=np.int64)
    lo = np.concatenate([a[a % 3 == 0], a[a % 7 == 0], a[a % 11 == 0]])
    hi = lo + np.repeat([1, 5, 16], [np.sum(a % 3 == 0), np.sum(a % 7 == 0), np.sum(a % 11 == 0)])
    lo, hi = lo[hi < n], hi[hi < n]
    i, j = np.concatenate([lo, hi]), np.concatenate([hi, lo])
    order = np.lexsort((j, i))
    st["nbr"] = j[order].astype(np.int32)
    st["nbr_off"] = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))]).astype(np.int32)
    return st


def _check(n, dim, precision, seed):
    sim = ca.Simulator(ca.Config(dim=dim, num_start=n, precision=precision, seed=1))
    st = _state(n, dim, precision == ca.PREC_MIXED, seed)
    sim.set_state(st, sim.scalars())
    for _ in range(2):
        out, sc = sim.get_state()
        assert sc["count"] == n
        for k, a in st.items():
            assert np.array_equal(out[k], a), k
    sim.close()


# one tile of a chunk's kernel and its neighbours, a field cut by a chunk's end
# (from 1e4 on), more chunks than slots and helpers (3e5)
@pytest.mark.parametrize("n", [33, 1023, 1025, 10007, 43691, 300001])
@pytest.mark.parametrize("dim,precision", [(2, 0), (3, 1), (3, 0)])
def test_written_state_comes_back(n, dim, precision):
    _check(n, dim, precision, n + dim)


def test_threads_read_at_once():
    failed = []

    def work(k):
        try:
            _check(20000 + 1001 * k, 2 + k % 2, k // 2 % 2, k)
        except BaseException as e:  # noqa: B036 (reported below)
            failed.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed


@pytest.mark.parametrize("precision", [0, 1])
def test_attempt_outputs_of_many_chunks(precision):
    """Each bubble's corrected position is x + dt / 2 (v + vp): three fields of
    the read-back and two of the state, of the same bubble."""
    sim = ca.Simulator(ca.Config(dim=3, num_start=200001, precision=precision, seed=3))
    ip = ca.IntegrationParams()
    sim.integrate(ip)
    st, sc = sim.get_state()
    sim.step(ip)
    at = sim.get_attempt()
    want = st["x"][:3] + 0.5 * sc["dt"] * (st["v"][:3] + at["vp"][:3])
    # three roundings of values no larger than these
    size = np.abs(st["x"][:3]) + sc["dt"] * (np.abs(st["v"][:3]) + np.abs(at["vp"][:3]))
    assert np.all(np.abs(at["xc"][:3] - want) <= 4 * 2.0 ** -53 * size)
    assert np.array_equal(at["del"] != 0, at["xc"][3] <= sc["min_rad"])
    sim.close()
