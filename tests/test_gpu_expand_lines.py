"""A forward on either side of the lines up to which it makes A = B theta in its own
blocks: the same A and the same points as for more thetas than that takes."""
import pytest
import torch

from libcpab_amd import Cpab
from libcpab_amd import _native as N
from libcpab_amd.pytorch import hip_ops as H

pytestmark = pytest.mark.gpu


# entries of B: 1984 and 2112 (1D), 7344 and 13248, 2880 and 8640
@pytest.mark.parametrize("nc", [[32], [33], [3, 3], [4, 3], [2, 2, 1], [3, 2, 1]])
def test_either_side_of_the_lines(cuda, nc):
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=True)
    L, dev, n = N.lib(), H.device_tess(T.params, cuda), 260
    gen = torch.Generator().manual_seed(6)
    theta = (torch.randn(n, dev.d, generator=gen) * 0.3).to(cuda)
    pts = torch.rand(len(nc), 200, generator=gen).to(cuda)

    def forward(th):
        A, out = dev.new_A(th).fill_(float("nan")), torch.empty(th.shape[0], len(nc), 200, device=cuda)
        N.check(L.cpab_transform_fwd_keep(dev.ref, H._ptr(th), th.shape[0], H._ptr(pts), 200, 0, None, 1.0, H._ptr(out),
                                          None, H._ptr(A), 4 * A.numel(), H._stream(cuda)))
        return A, out

    A, out = forward(theta)
    want = dev.new_A(theta)
    N.check(L.cpab_theta_to_A(dev.ref, H._ptr(theta), n, H._ptr(want), H._stream(cuda)))
    assert torch.equal(A, want)
    for k in (0, n - 1):
        A1, out1 = forward(theta[k:k + 1].contiguous())
        assert torch.equal(A1[0], A[k]) and torch.equal(out1[0], out[k])
