"""The fixed-step scheme's maps and exponentials on both sides of the rule that
takes them in one launch or two: the same bits."""
import pytest
import torch

from libcpab_amd import Cpab
from libcpab_amd import _native as N
from libcpab_amd.pytorch import hip_ops as H

pytestmark = pytest.mark.gpu


def _expand(dev, theta, steps):
    As = dev.new_A(theta).fill_(float("nan"))
    trels = As.clone()
    N.check(N.lib().cpab_ref_expand(dev.ref, H._ptr(theta), theta.shape[0], steps, H._ptr(As), H._ptr(trels),
                                    H._stream(theta.device)))
    return As, trels


# one theta at a time is one launch where B has at most 2^13 entries, n together two:
# 257 blocks of 2D and 3D maps, 1025 of 1D ones; a block's last piece whole and not
@pytest.mark.parametrize("nc,n", [([10], 1025), ([40], 513), ([2, 2], 257), ([3, 3], 129), ([1, 1, 1], 257)])
def test_thetas_alone_and_together(cuda, nc, n):
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=nc != [1, 1, 1])
    dev = H.device_tess(T.params, cuda)
    assert dev.nC * len(nc) * (len(nc) + 1) * dev.d <= 1 << 13
    theta = torch.randn(n, dev.d, generator=torch.Generator().manual_seed(8)).to(cuda)
    As, trels = _expand(dev, theta, 50)
    for k in (0, 1, n // 2, n - 1):
        A1, t1 = _expand(dev, theta[k:k + 1].contiguous(), 50)
        assert torch.equal(A1[0], As[k]) and torch.equal(t1[0], trels[k])


# B beyond 2^13 entries: against FP64, and the exponentials of the maps by themselves
@pytest.mark.parametrize("nc,n", [([70], 3), ([8, 8], 1), ([2, 2, 2], 5), ([3, 3, 3], 2)])
def test_large_bases(cuda, nc, n):
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=True)
    dev = H.device_tess(T.params, cuda)
    theta = torch.randn(n, dev.d, generator=torch.Generator().manual_seed(9)).to(cuda)
    As, trels = _expand(dev, theta, 32)
    B = dev.B.double()
    size = theta.double().abs() @ B.t().abs().contiguous()
    assert ((As.double() - theta.double() @ B.t().contiguous()).abs() <= (dev.d + 2) * 2.0 ** -24 * size + 1e-30).all()
    want = torch.empty_like(As)
    N.check(N.lib().cpab_expm_affine(H._ptr(As), n * dev.nC, len(nc), 1 / 32, H._ptr(want), H._stream(cuda)))
    assert torch.equal(trels, want)
