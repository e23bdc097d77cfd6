"""Sizes of the fixed-step gradient's workspace up to the largest point count."""
import pytest

from libcpab_amd import _native as N


@pytest.mark.parametrize("n", [1, 7])
@pytest.mark.parametrize("nP", [64, 65, 4096 * 64 + 1, (1 << 31) - 64, (1 << 31) - 63, (1 << 31) - 1])
def test_blocks_of_sixty_four_points_up_to_4096(n, nP):
    nc = N.int3([2, 2])
    blocks = min((nP + 63) // 64, 4096 // n)
    assert N.lib().cpab_ref_grad_workspace_bytes(2, nc, n, nP, 50) == n * blocks * 16 * 6 * 4
