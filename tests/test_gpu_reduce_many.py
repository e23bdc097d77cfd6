"""dL/dtheta of a thousand thetas with few rows of partials each, against one call
per theta, which reduces in another order: at most some 230 FP32 additions on the
way of any term, so 1.4e-5 of the terms' absolute sum, taken as three times the
largest entry."""
import pytest
import torch

from libcpab_amd import Cpab

pytestmark = pytest.mark.gpu


# d = nC - 1 in 1D: below, at and above a block's 64 columns; D below and above 64 rows; thetas that do not fill the
# last block; one and several rows; a base beyond 2^15 entries
@pytest.mark.parametrize("nc,n,nP", [([2], 1024, 200), ([50], 4099, 1024), ([65], 1025, 300), ([66], 1100, 300),
                                     ([30], 1024, 4000), ([5, 5], 1024, 900)])
def test_many_thetas_match_single_calls(cuda, nc, n, nP):
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=True)
    gen = torch.Generator().manual_seed(6)
    theta = (torch.randn(n, T.get_theta_dim(), generator=gen) * 0.3).to(cuda).requires_grad_(True)
    pts = torch.rand(len(nc), nP, generator=gen).to(cuda)
    up = (torch.rand(n, len(nc), nP, generator=gen) + 0.2).to(cuda)
    got, = torch.autograd.grad(T.transform_grid(pts, theta), theta, up)
    again, = torch.autograd.grad(T.transform_grid(pts, theta), theta, up)
    assert torch.equal(got, again)
    for k in (0, 1, n // 2, n - 1):
        th = theta[k:k + 1].detach().requires_grad_(True)
        want, = torch.autograd.grad(T.transform_grid(pts, th), th, up[k:k + 1])
        assert float((got[k] - want[0]).abs().max()) <= 4e-5 * float(want.abs().max())
