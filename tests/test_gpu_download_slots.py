"""get_state on both sides of the 32 MiB from which states are downloaded
through pinned slots of 2 MiB (capi.cpp, download), with whole slots, a last
chunk of 40 bytes and one that is 40 bytes short: the caller's own bits, in a
context's first read, its later ones, and from another thread than the one
that made the context."""
import threading

import numpy as np
import pytest

from finess_amd import BC_PERIODIC, Solver, default_params

pytestmark = pytest.mark.gpu

LARGE, SLOT = 32 << 20, 2 << 20
# (mx + 6, my + 6) and what its 40 bytes a cell are
SHAPES = [((820, 1023), lambda n: LARGE - 40 < n < LARGE), ((397, 2113), lambda n: LARGE < n < LARGE + 40),
          ((1024, 1024), lambda n: n % SLOT == 0), ((17, 61681), lambda n: n % SLOT == 40),
          ((1023, 1025), lambda n: n % SLOT == SLOT - 40)]


@pytest.mark.parametrize("shape,what", SHAPES)
def test_round_trip(shape, what):
    p = default_params(mx=shape[0] - 6, my=shape[1] - 6, bc=[BC_PERIODIC] * 4)
    q = np.random.default_rng(shape[1]).random(p.shape_q())
    g = p.mbc
    q = np.ascontiguousarray(np.pad(q[g:-g, g:-g], ((g, g), (g, g), (0, 0)), mode="wrap"))
    assert q.shape == shape + (5,) and what(q.nbytes)
    got = []
    with Solver(p) as s:
        s.set_state(q)
        got.append(s.get_state()[0])
        t = threading.Thread(target=lambda: got.append(s.get_state()[0]))
        t.start()
        t.join()
        s.set_state(q + 1)
        got.append(s.get_state()[0] - 1)
    assert len(got) == 3 and all(np.array_equal(r, q) for r in got[:2])
    assert np.array_equal(got[2], (q + 1) - 1)
