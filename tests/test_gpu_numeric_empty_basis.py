"""method='numeric' on a tessellation whose basis has no columns (one cell whose two
ends are held): every theta is the identity."""
import pytest
import torch

from libcpab_amd import Cpab

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3])
def test_no_parameters_is_the_identity(cuda, n):
    T = Cpab([1], backend="pytorch", device="gpu", zero_boundary=True)
    assert T.get_theta_dim() == 0
    T.set_solver_params(nstepsolver=20, method="numeric")
    grid = T.uniform_meshgrid([33])
    out = T.transform_grid(grid, torch.zeros(n, 0, device=cuda))
    assert torch.equal(out, grid[None].expand(n, 1, 33))
