"""A = B theta on both sides of the rule that picks its kernel, at the edges of
their tiles: every entry is its products added in one order, within (d + 2)
roundings of the FP64 value."""
import pytest
import torch

from libcpab_amd import Cpab
from libcpab_amd import _native as N
from libcpab_amd.pytorch import hip_ops as H

pytestmark = pytest.mark.gpu


# products n * D * d: below 2^20 (a thread per entry) and above, with 1, 2, 4 and 8 thetas a wave; d below, at and
# above a piece of 64 columns; D whole and not whole tiles of 64 rows
@pytest.mark.parametrize("nc,n", [([2], 1), ([65], 3), ([66], 200), ([70], 5000), ([3, 3], 300), ([4, 4], 3000),
                                  ([8, 8], 65), ([2, 2, 2], 1001), ([3, 3, 3], 17)])
def test_expansion_matches_fp64(cuda, nc, n):
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=True)
    dev = H.device_tess(T.params, cuda)
    nd, d = len(nc), T.get_theta_dim()
    theta = torch.randn(n, d, generator=torch.Generator().manual_seed(2)).to(cuda)
    A = dev.new_A(theta).fill_(float("nan"))
    N.check(N.lib().cpab_theta_to_A(dev.ref, H._ptr(theta), n, H._ptr(A), H._stream(theta.device)))
    col = torch.tensor([1.0 / c for c in nc] + [1.0], dtype=torch.float64, device=cuda)
    scale = (torch.tensor(nc, dtype=torch.float64, device=cuda)[:, None] * col[None, :]).reshape(-1)
    scale = scale.repeat(dev.nC)
    B = dev.B.double()
    want = theta.double() @ B.t().contiguous() * scale
    size = theta.double().abs() @ B.t().abs().contiguous() * scale
    assert ((A.double() - want).abs() <= (d + 2) * 2.0 ** -24 * size + 1e-30).all()
