"""More points in one call than the saved state's 32-bit offsets reach: the
forward with gradients is the forward without, bit for bit, and dL/dtheta the
recomputed one."""
import pytest
import torch

from libcpab_amd import Cpab

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,out", [([2, 2], [32768, 32769]), ([1, 1, 1], [1024, 1024, 1025])])
def test_beyond_the_saved_state(cuda, nc, out):
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=False)
    gen = torch.Generator(device=cuda).manual_seed(3)
    theta = torch.randn(1, T.get_theta_dim(), generator=gen, device=cuda) * 0.1
    data = torch.rand(1, 1, *([24] * len(nc)), generator=gen, device=cuda)
    up = torch.rand(1, 1, *out, generator=gen, device=cuda)
    plain = T.transform_data(data, theta, out)
    leaf = theta.clone().requires_grad_()
    got = T.transform_data(data, leaf, out)
    assert torch.equal(got.detach(), plain)
    g, = torch.autograd.grad(got, leaf, up)
    del got
    T.params.store_jacobian = False
    again = T.transform_data(data, leaf, out)
    want, = torch.autograd.grad(again, leaf, up)
    assert torch.isfinite(g).all() and torch.equal(g, want)
