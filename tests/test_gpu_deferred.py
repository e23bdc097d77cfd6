"""The 3D backward that lets points wait in LDS between chunks gives the gradient
of the one that runs each point to its end (taken where dL/ddata is asked for
too), over trajectories of one to many chunks, with whole and partial tiles."""
import pytest
import torch

from libcpab_amd import Cpab

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,size,n,scale", [([3, 3, 3], [64, 64, 64], 16, 0.2), ([3, 3, 3], [61, 67, 66], 17, 0.8),
                                             ([1, 2, 1], [70, 65, 64], 16, 0.5)])
def test_deferred_points_give_the_same_gradient(cuda, nc, size, n, scale):
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=True)
    gen = torch.Generator().manual_seed(7)
    theta = (torch.randn(n, T.get_theta_dim(), generator=gen) * scale).to(cuda).requires_grad_(True)
    ax = [torch.linspace(0, 1, s) for s in size]
    data = (ax[0][:, None, None] + 2 * ax[1][None, :, None] - ax[2][None, None, :]).expand([n, 1] + size)
    data = data.contiguous().to(cuda).requires_grad_(True)
    up = torch.rand([n, 1] + size, generator=gen).to(cuda)
    one, = torch.autograd.grad(T.transform_data(data, theta, size), theta, up)
    two, _ = torch.autograd.grad(T.transform_data(data, theta, size), (theta, data), up)
    again, = torch.autograd.grad(T.transform_data(data, theta, size), theta, up)
    assert torch.equal(one, again)
    # the same terms in another order: at most some 230 FP32 additions on the way of any of them (wave folds, LDS
    # accumulator, rows, B^T), so 1.4e-5 of the terms' absolute sum, taken as three times the largest entry
    assert float((one - two).abs().max()) <= 4e-5 * float(two.abs().max())
