"""The 1D run kernel where its waves' chunks of 31 cells do not fill the last
round, and at the limit of the kinds with pow: bit for bit the host
controller's launches (see test_gpu_run1d)."""
import pytest

from finess_amd import BC_EXTRAP, BC_PERIODIC, BC_REFLECT, WENO_FD, WENO_Z
from test_gpu_run1d import _problem, _same

pytestmark = pytest.mark.gpu

# one cell less and more than 16, 32 and 64 chunks, one and two chunks of the last round, its first and last wave
SIZES = [496, 497, 527, 528, 558, 961, 962, 992, 993, 1488, 1489, 1536, 1537, 1984, 1985, 2480, 2481]


@pytest.mark.parametrize("kw", [dict(), dict(weno_version=WENO_FD), dict(power_param=1.5),
                                dict(weno_version=WENO_Z, power_param=3.0)])
@pytest.mark.parametrize("mx", SIZES)
def test_partial_rounds(mx, kw):
    bc = [[BC_PERIODIC] * 4, [BC_REFLECT, BC_EXTRAP] + [BC_PERIODIC] * 2][mx % 2]
    p, q, aux = _problem(mx, bc=bc, **kw)
    _same(p, q, aux, 7.3 * 0.4 / mx / 1.5)
