"""The primitive-record tile on the workgroup's real LDS layout, whose arrays
overlay each other (stage_prim.h: the y fluxes take the records' place, with
Lax-Wendroff the x fluxes F's), phase by phase on the CPU against the oracle:
both forms of the tile, both physics, Runge-Kutta and Lax-Wendroff, every
reconstruction.  Tolerance as in test_emu_prim, 5e-13 of max |L| per field."""
import ctypes

import numpy as np
import pytest

import orc
from finess_amd import BC_EXTRAP, BC_PERIODIC, BC_REFLECT, TS_LXW, WENO_FD, WENO_Z, Params, problems

PD = ctypes.POINTER(ctypes.c_double)
KINDS = [dict(), dict(power_param=1.5), dict(weno_version=WENO_Z), dict(weno_version=WENO_Z, power_param=3.0),
         dict(weno_version=WENO_FD)]
MIXED = [BC_EXTRAP, BC_PERIODIC, BC_REFLECT, BC_REFLECT]


def _planes(a):
    return np.ascontiguousarray(np.moveaxis(a, -1, 0))


@pytest.mark.parametrize("two", [0, 1])
@pytest.mark.parametrize("lxw", [0, 1])
@pytest.mark.parametrize("what", ["euler", "euler_w", "shallow_water"])
@pytest.mark.parametrize("kw", KINDS)
def test_overlay(kw, what, lxw, two):
    rng = np.random.default_rng(4)
    kw = dict(kw, bc=MIXED)
    if lxw:
        kw.update(time_stepping_method=TS_LXW, mbc=5, time_order=3)
    if what == "shallow_water":
        p, q, _ = problems.sw_bump(nx=37, ny=35, **kw)
        q[..., 1:] = 0.1 * rng.random(q.shape[:-1] + (2,))
    else:
        p, q, _ = problems.riemann4(mx=37, my=35, **kw)
        q[..., 0] *= 1 + 0.05 * rng.random(q.shape[:-1])
        if what == "euler_w":
            q[:, :18, 3] = 0.2 * rng.random((q.shape[0], 18))
            q[..., 4] += 0.5 * q[..., 3] ** 2 / q[..., 0]
    orc.set_bnd(p, q)
    q = np.ascontiguousarray(q)
    F = G = None
    if lxw:
        F0, G0 = orc.integrated_r(p, 2e-3, q)
        L0, sm = np.zeros(p.shape_q()), np.zeros(p.shape_smax())
        orc.oracle().orc_construct_lxw_l(ctypes.byref(p), orc.ptr(q), orc.ptr(np.ones(p.shape_aux())), orc.ptr(F0),
                                         orc.ptr(G0), orc.ptr(L0), orc.ptr(sm))
        e = p.mbc - 3  # the extended grid has three ghosts
        F, G = (_planes(a[e:-e, e:-e]) for a in (F0, G0))
    else:
        L0, _ = orc.construct_l(p, q)
    lib = orc.emu()
    lib.emu_prim_overlay.argtypes = [ctypes.POINTER(Params), PD, PD, PD, ctypes.c_int, PD]
    planes = _planes(orc.interior(p, q))
    L = np.full_like(planes, np.nan)
    lib.emu_prim_overlay(ctypes.byref(p), orc.ptr(planes), orc.ptr(F), orc.ptr(G), two, orc.ptr(L))
    ref = np.moveaxis(orc.interior(p, L0), -1, 0)
    scale = np.abs(ref).max(axis=(1, 2), keepdims=True)
    assert scale[0] > 0 and np.all(np.abs(L - ref) <= 5e-13 * np.where(scale > 0, scale, 1.0))
