"""1D forwards of many points per thread read whole-cell crossings from a table;
single thetas do not.  Both give the same bits: the table's entries come from the
operations of a point that starts on the edge."""
import pytest
import torch

from libcpab_amd import Cpab

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,zb", [(2, True), (50, True), (64, True), (129, True), (5, False), (100, False)])
@pytest.mark.parametrize("scale", [0.5, 3.0])
def test_table_gives_the_same_bits(cuda, nc, zb, scale):
    T = Cpab([nc], backend="pytorch", device="gpu", zero_boundary=zb)
    gen = torch.Generator().manual_seed(5)
    n, nP = 4100, 1031  # 4 points per thread
    theta = (torch.randn(n, T.get_theta_dim(), generator=gen) * scale).to(cuda)
    theta[7] = 0.0
    pts = torch.cat([torch.linspace(-0.1, 1.1, 530), torch.arange(nc + 1) / nc, torch.rand(500 - nc, generator=gen)])
    pts = pts[None].to(cuda)
    data = torch.rand(n, 1, 64, generator=gen).to(cuda)
    many, warped = T.transform_grid(pts, theta), T.transform_data(data, theta, [nP])
    for k in (0, 7, 2048, n - 1):
        assert torch.equal(many[k], T.transform_grid(pts, theta[k:k + 1])[0])
        assert torch.equal(warped[k], T.transform_data(data[k:k + 1], theta[k:k + 1], [nP])[0])
