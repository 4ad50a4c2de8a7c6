"""Batch members with fewer cells than a periodic or reflecting side has ghosts
are refused before anything is allocated or launched (their ghosts would be
read from outside their planes); with extrapolation any size stays accepted.
Runs without a GPU, where an accepted batch ends with "no device"."""
import pytest

from finess_amd import BC_EXTRAP, BC_PERIODIC, BC_REFLECT, ERR_CONFIG, ERR_NODEVICE, Batch, FinessError, problems


def _create(sizes, bc):
    p = problems.sw_bump(nx=16, ny=16, bc=bc)[0]
    try:
        with Batch(p, sizes):
            return 0
    except FinessError as e:
        return e.code


@pytest.mark.parametrize("small", [1, 2])
@pytest.mark.parametrize("side", [0, 1, 2, 3])
@pytest.mark.parametrize("kind", [BC_PERIODIC, BC_REFLECT])
def test_small_member_refused(kind, side, small):
    bc = [BC_EXTRAP] * 4
    bc[side] = kind
    size = (small, 16) if side < 2 else (16, small)
    assert _create([(16, 16), size], bc) == ERR_CONFIG
    assert _create([(16, 16), size[::-1]], bc) in (0, ERR_NODEVICE)


def test_smallest_members_accepted():
    assert _create([(3, 16), (16, 3), (3, 3)], [BC_PERIODIC] * 2 + [BC_REFLECT] * 2) in (0, ERR_NODEVICE)
    assert _create([(1, 1), (2, 16)], [BC_EXTRAP] * 4) in (0, ERR_NODEVICE)
