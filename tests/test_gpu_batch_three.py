"""Three points a thread in the batched backward: 768-point tiles with dL/ddata in
bins where they cover few enough samples, and past that, against the
single-problem path."""
import pytest
import torch

from libcpab_amd import Cpab
from libcpab_amd.batch import CpabBatch

pytestmark = pytest.mark.gpu

# a 48 x 16 tile covers, per axis, its share of the samples and one more: 49 x 17 = 833
# at the same size (no bins), about 33 x 12 at two thirds, 25 x 9 at a half; 44 x 17 =
# 748 and 46 x 17 = 782 lie on either side of the 767 that fit
SIZES = [([64, 64], [64, 64]), ([43, 43], [64, 64]), ([33, 17], [97, 70]), ([86, 64], [96, 64]), ([90, 64], [96, 64]),
         ([9, 200], [61, 50]), ([5, 5], [48, 16])]


@pytest.mark.parametrize("channels", [1, 3, 4, 5])
def test_three_points_a_thread(cuda, channels):
    g = torch.Generator().manual_seed(12)
    T = Cpab([3, 2], backend="pytorch", device="gpu", zero_boundary=True)
    b = CpabBatch([(T, channels, s, o) for s, o in SIZES], device=cuda, save=True, ppt=3, blocks=512)
    # small enough that the tiles' footprints stay as they are without a warp
    for i, (s, o) in enumerate(SIZES):
        b.theta_views[i].copy_(torch.randn(T.get_theta_dim(), generator=g) * 0.02)
        b.data_views[i].copy_(torch.rand([channels] + s, generator=g))
        b.grad_out_views[i].copy_(torch.randn([channels] + o, generator=g))
    b.forward()
    b.backward()
    for i, (s, o) in enumerate(SIZES):
        th = b.theta_views[i].clone()[None].requires_grad_(True)
        da = b.data_views[i].clone()[None].requires_grad_(True)
        out = T.transform_data(da, th, o)
        gth, gda = torch.autograd.grad(out, (th, da), b.grad_out_views[i][None])
        # orders of summation differ: roundings of sums of n terms, n the points of a sample
        # or of the problem
        n_da, n = (o[0] / s[0] + 2) * (o[1] / s[1] + 2) * 4, o[0] * o[1]
        top = b.grad_out_views[i].abs().max()
        assert torch.equal(b.out_views[i], out[0])
        assert (b.grad_data_views[i] - gda[0]).abs().max() <= 2 * n_da * 2.0 ** -24 * n_da * top
        assert (b.grad_theta_views[i] - gth[0]).abs().max() <= 64 * n ** 0.5 * 2.0 ** -24 * gth[0].abs().max() + 1e-6
