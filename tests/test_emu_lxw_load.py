"""The Lax-Wendroff flux kernel's load phase with the workgroup's size given
(lxw_phase_load with nthreads): any number of threads up to the tile's cells
leaves the same fluxes, bit for bit, as one thread per cell."""
import ctypes

import numpy as np
import pytest

import orc
from finess_amd import TS_LXW, Params, problems

PD = ctypes.POINTER(ctypes.c_double)


@pytest.mark.parametrize("nthreads", [1, 100, 256])
def test_load_with_fewer_threads(nthreads):
    p, q, _ = problems.riemann4(mx=13, my=35, time_stepping_method=TS_LXW, mbc=5, time_order=3)
    orc.set_bnd(p, q)
    q = np.ascontiguousarray(q)
    lib = orc.emu()
    lib.emu_integrated_threads.argtypes = [ctypes.POINTER(Params), ctypes.c_double, PD, ctypes.c_int, PD, PD]
    F0, G0, F1, G1 = (np.zeros_like(q) for _ in range(4))
    lib.emu_construct_integrated_r(ctypes.byref(p), 1e-3, orc.ptr(q), orc.ptr(F0), orc.ptr(G0))
    lib.emu_integrated_threads(ctypes.byref(p), 1e-3, orc.ptr(q), nthreads, orc.ptr(F1), orc.ptr(G1))
    assert np.abs(F0).max() > 0 and np.array_equal(F0, F1) and np.array_equal(G0, G1)
