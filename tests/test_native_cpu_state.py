"""The range of the saved state: in 2D and 3D the chunk log and the rows beside it
are addressed by 32-bit byte offsets, so from 2^29 points per theta on the calls
keep none (the size functions say 0, nothing is launched here)."""
import pytest

from libcpab_amd import _native as N

LIMIT = 1 << 29


@pytest.mark.parametrize("ndim,saved,jac", [(2, 9, 7), (3, 15, 12)])
def test_no_state_from_two_to_the_29_points_on(ndim, saved, jac):
    L = N.lib()
    for n in (1, 3):
        assert L.cpab_saved_floats(ndim, n, LIMIT - 1) == n * saved * (LIMIT - 1)
        assert L.cpab_jac_floats(ndim, n, LIMIT - 1) == n * jac * (LIMIT - 1)
        for nP in (LIMIT, 2 * LIMIT + 5, (1 << 31) - 1):
            assert L.cpab_saved_floats(ndim, n, nP) == 0
            assert L.cpab_jac_floats(ndim, n, nP) == 0


def test_signals_keep_state_at_any_length():
    L = N.lib()
    assert L.cpab_saved_floats(1, 2, LIMIT) == 2 * 2 * LIMIT
    assert L.cpab_jac_floats(1, 2, LIMIT) == 2 * LIMIT
