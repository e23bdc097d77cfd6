"""The table of whole-cell crossings at the edges of its range, in both directions:
up to 512 cells and 64 for each point of a thread.  Points are the same bits as a
single theta's, which has no table; its gradient's terms are too, added in another
order (some 230 FP32 additions, so 1.4e-5 of their absolute sum, taken as three
times the gradient's norm)."""
import pytest
import torch

from libcpab_amd import Cpab

pytestmark = pytest.mark.gpu


# 8 points a thread: 512 cells take the table, 513 do not; 2: 128 and 129
@pytest.mark.parametrize("nc,n,nP", [(3, 4100, 1031), (512, 4100, 1031), (513, 4100, 1031), (128, 1200, 2000),
                                     (129, 1200, 2000)])
def test_table_in_both_directions(cuda, nc, n, nP):
    T = Cpab([nc], backend="pytorch", device="gpu", zero_boundary=True)
    gen = torch.Generator().manual_seed(7)
    theta = (torch.randn(n, T.get_theta_dim(), generator=gen) * min(0.5, 20.0 / nc)).to(cuda).requires_grad_(True)
    pts = torch.cat([torch.arange(nc + 1) / nc, torch.rand(nP - nc - 1, generator=gen)])[None].to(cuda)
    data = torch.linspace(0, 1, 64).repeat(n, 1, 1).to(cuda)  # a ramp: its slope is the upstream's factor
    up = (torch.rand(n, 1, nP, generator=gen) + 0.2).to(cuda)

    def passes(th, rows):
        grid = T.transform_grid(pts, th)
        warped = T.transform_data(data[rows], th, [nP])
        return [grid, warped] + [torch.autograd.grad(o, th, up[rows])[0] for o in (grid, warped)]

    many = passes(theta, slice(0, n))
    for k in (0, n // 2, n - 1):
        one = passes(theta[k:k + 1].detach().requires_grad_(True), slice(k, k + 1))
        assert torch.equal(many[0][k], one[0][0]) and torch.equal(many[1][k], one[1][0])
        for got, want in zip(many[2:], one[2:]):
            assert float((got[k] - want[0]).abs().max()) <= 4.2e-5 * float(want.norm())
