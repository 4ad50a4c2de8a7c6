"""finess_construct_l_planes_noalloc after a call that failed: the wave-speed
maxima of a failed call must not reach the next one.  The failure is an error
left unread on the calling thread (an invalid hipSetDevice, refused by the
runtime on the host), which the call's own launch check then finds."""
import ctypes

import numpy as np
import pytest

import orc
from finess_amd import load_library, problems
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("global_alpha", [0, 1])
def test_failed_call_leaves_no_speeds(global_alpha):
    lib, hip = load_library(), _Hip()
    p, q, _ = problems.riemann4(mx=40, my=36, global_alpha=global_alpha)
    slow = np.ascontiguousarray(np.moveaxis(orc.interior(p, q), -1, 0))
    fast = slow.copy()
    fast[1] += 20.0 * fast[0]  # u + 20
    fast[4] += 20.0 * slow[1] + 200.0 * fast[0]
    try:
        qs, qf, Ld = hip.upload(slow), hip.upload(fast), hip.upload(np.zeros(slow.shape))

        def call(qd):
            sd = hip.upload(np.full(2, np.nan))
            rc = lib.finess_construct_l_planes_noalloc(ctypes.byref(p), qd, Ld, sd, None)
            assert hip.rt.hipDeviceSynchronize() == 0
            return rc, hip.download(sd, (2,))

        rc, s0 = call(qs)
        assert rc == 0
        assert hip.rt.hipSetDevice(10000) != 0
        rc, _ = call(qf)
        print("call with an unread error on its thread:", rc)
        rc, s1 = call(qs)
        assert rc == 0 and np.array_equal(s0, s1), (s0, s1)
        rc, s2 = call(qf)
        assert rc == 0 and s2[0] > s0[0] + 15.0
    finally:
        hip.close()
