"""dL/dtheta of thousands of thetas where the reduction takes four and eight thetas
a wave, and five and six rows of partials of a large base, against one call per
theta: at most some 230 FP32 additions on the way of any term, so 1.4e-5 of the
terms' absolute sum, taken as three times the gradient's norm."""
import pytest
import torch

from libcpab_amd import Cpab

pytestmark = pytest.mark.gpu


# [8, 8] (four column blocks): from 2041 thetas on four a wave, from 4065 on eight; one column block: eight from
# 16353 on.  None fills the last block.
@pytest.mark.parametrize("nc,n,nP", [([8, 8], 2051, 300), ([8, 8], 4101, 130), ([20], 16390, 40), ([5, 5], 1100, 1100),
                                     ([5, 5], 1101, 1500)])
def test_many_thetas_match_single_calls(cuda, nc, n, nP):
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=True)
    gen = torch.Generator().manual_seed(6)
    theta = (torch.randn(n, T.get_theta_dim(), generator=gen) * 0.3).to(cuda).requires_grad_(True)
    pts = torch.rand(len(nc), nP, generator=gen).to(cuda)
    up = (torch.rand(n, len(nc), nP, generator=gen) + 0.2).to(cuda)
    got, = torch.autograd.grad(T.transform_grid(pts, theta), theta, up)
    for k in (0, 1, n // 2, n - 3, n - 2, n - 1):
        th = theta[k:k + 1].detach().requires_grad_(True)
        want, = torch.autograd.grad(T.transform_grid(pts, th), th, up[k:k + 1])
        assert float((got[k] - want[0]).abs().max()) <= 4.2e-5 * float(want.norm())
