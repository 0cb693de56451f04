"""GPU test of reading neighbour lists of more than 2^31 entries in all: their
length is compared with the caller's room, and every entry lands in its place."""
import ctypes

import numpy as np
import pytest

import cubble_amd as ca

pytestmark = pytest.mark.gpu


def test_more_than_two_to_the_31_entries():
    """46,400 bubbles of which each touches every other one: bubble i's list is
    0, .., i - 1, i + 1, .."""
    n = 46400
    total = n * (n - 1)
    assert total > 2 ** 31
    sim = ca.Simulator(ca.Config(dim=2, num_start=n, seed=1))
    st, sc = sim.get_state()
    st["x"][3] = sc["max_r_cell"] = sum(sc["interval"])
    st["nbr_off"][:] = 0
    st["nbr"] = np.zeros(0, np.int32)
    sim.set_state(st, sc)
    sim.search_neighbors()
    print(f"searched, {total} entries", flush=True)

    v = ca._StateView()
    off = np.zeros(n + 1, np.int32)
    nbr = np.zeros(16, np.int32)
    v.nbr_off, v.nbr, v.nbr_cap = off.ctypes.data, nbr.ctypes.data, 16
    # no room: refused, and nothing written past the room
    rc = ca.lib().cubble_get_state(sim._h, ctypes.byref(v))
    assert rc != ca.OK and not nbr.any()
    assert np.array_equal(off.view(np.uint32),
                          (np.arange(n + 1, dtype=np.uint64) * (n - 1)).astype(np.uint32))
    del nbr
    room = np.empty(total, np.int32)
    v.nbr, v.nbr_cap = room.ctypes.data, total
    assert ca.lib().cubble_get_state(sim._h, ctypes.byref(v)) == ca.OK
    print("read", flush=True)
    every = np.arange(n, dtype=np.int32)
    for i in (0, 1, 1023, 1024, n // 2, 46283, 46284, n - 2, n - 1):
        assert np.array_equal(room[i * (n - 1):(i + 1) * (n - 1)], np.delete(every, i)), i
    sim.close()
