"""The fixed-step gradient with nearly 2^31 points: the last step of a block's walk
over them ends beyond 2^31.  dL/dtheta is the sum of the two halves'."""
import pytest
import torch

from libcpab_amd import Cpab

pytestmark = pytest.mark.gpu


def test_gradient_of_the_longest_signal(cuda):
    T = Cpab([2], backend="pytorch", device="gpu", zero_boundary=False)
    T.set_solver_params(nstepsolver=2, method="numeric")
    gen = torch.Generator(device=cuda).manual_seed(5)
    theta = torch.randn(1, T.get_theta_dim(), generator=gen, device=cuda) * 0.1
    nP = (1 << 31) - 4096
    x = torch.rand(1, nP, generator=gen, device=cuda)
    up = torch.rand(1, 1, nP, generator=gen, device=cuda)

    def grad(lo, hi):
        leaf = theta.clone().requires_grad_()
        out = T.transform_grid(x[:, lo:hi], leaf)
        return torch.autograd.grad(out, leaf, up[..., lo:hi])[0].double()

    whole, halves = grad(0, nP), grad(0, nP // 2) + grad(nP // 2, nP)
    # 8192 FP32 additions into a wave's sum, 4096 waves' sums
    assert (whole - halves).abs().max() <= 2 * (8192 + 16) * 2.0 ** -24 * halves.abs().max()
