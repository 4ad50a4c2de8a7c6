"""WENO-Z at power 2 on states of any size.  The scheme is homogeneous in the
conserved variables once eps is negligible (L of c q is c L of q), and its
weights take ratios of indicators, which go with c^2: three of them multiplied
overflow from c = 1e51 on.  (Noise in every field: where a stencil is flat but
for one jump, the ratio over eps itself overflows when squared.)  Bounds: those
of test_emu_prim for one evaluation, 5e-13 of max |L| per field."""
import ctypes

import numpy as np
import pytest

import orc
from finess_amd import BC_PERIODIC, WENO_Z, Params, problems

PD = ctypes.POINTER(ctypes.c_double)


def _state(size):
    p, _, _ = problems.riemann4(mx=23, my=17, weno_version=WENO_Z, bc=[BC_PERIODIC] * 4)
    rng = np.random.default_rng(2)
    rho, u, v, w, pr = (1 + 0.2 * rng.random(p.shape_q()[:-1]) for _ in range(5))
    e = pr / (p.gamma - 1) + 0.5 * rho * (u * u + v * v + w * w)
    q = np.stack([rho, rho * u, rho * v, rho * w, e], axis=-1)
    q *= size
    orc.set_bnd(p, q)
    return p, q


@pytest.mark.parametrize("two", [0, 1])
@pytest.mark.parametrize("size", [1e-10, 1.0, 1e45, 1e52, 1e70, 1e100])
def test_euler_z_sizes(size, two):
    p, q = _state(size)
    lib = orc.emu()
    lib.emu_prim_l.argtypes = [ctypes.POINTER(Params), PD, ctypes.c_int, PD, PD, PD]
    L0, _ = orc.construct_l(p, q)
    planes = np.ascontiguousarray(np.moveaxis(orc.interior(p, q), -1, 0))
    L, sx, sy = np.zeros_like(planes), np.zeros((p.mx + 1, p.my)), np.zeros((p.mx, p.my + 1))
    lib.emu_prim_l(ctypes.byref(p), orc.ptr(planes), two, orc.ptr(L), orc.ptr(sx), orc.ptr(sy))
    ref = np.moveaxis(orc.interior(p, L0), -1, 0)
    scale = np.abs(ref).max(axis=(1, 2), keepdims=True)
    assert np.all(np.isfinite(ref)) and scale[0] > 0
    assert np.all(np.abs(L - ref) <= 5e-13 * np.where(scale > 0, scale, 1.0))
