"""The FP32 Lax-Wendroff stage with its stencil fluxes in LDS (grids of 2.8
million cells and more) against the stage that reads them from memory: a
periodic state repeated over the large grid steps like the one on the small
grid, bit for bit (the same operations in the same order)."""
import numpy as np
import pytest

from finess_amd import BC_PERIODIC, PREC_FP32, Solver, problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [2, 3])
def test_repeated_state(order):
    shape, rep = (187, 188), (9, 9)  # 1683 x 1692: partial tiles at both edges

    def solve(mx, my, q):
        p, q0, _ = problems.kelvin_helmholtz(mx=mx, my=my, time_order=order, precision=PREC_FP32,
                                             xlow=0.0, xhigh=float(mx), ylow=0.0, yhigh=float(my))
        assert list(p.bc) == [BC_PERIODIC] * 4 and p.dx == 1.0 and p.dy == 1.0
        g = p.mbc
        if q is None:
            q = q0[g:-g, g:-g].copy()
            q[..., 0] *= 1.0 + 0.1 * np.random.default_rng(3).random(q.shape[:-1])
        with Solver(p) as s:
            s.set_state(np.pad(q, ((g, g), (g, g), (0, 0)), mode="wrap"))
            s.run_fixed_steps(0.2, 2)
            return q, s.get_state()[0][g:-g, g:-g]

    q, small = solve(*shape, None)
    large = solve(shape[0] * rep[0], shape[1] * rep[1], np.tile(q, rep + (1,)))[1]
    assert np.abs(small - q).max() > 1e-3
    assert np.array_equal(large, np.tile(small, rep + (1,)))
