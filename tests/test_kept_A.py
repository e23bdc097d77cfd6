"""The transforms that keep A = B theta from the forward to the backward give,
bit for bit, what the entry points that make A in each direction give: the same
numbers come from the same kernels."""
import ctypes

import pytest
import torch

from libcpab_amd import Cpab
from libcpab_amd import _native as N
from libcpab_amd.pytorch import hip_ops as H


@pytest.mark.gpu
@pytest.mark.parametrize("nc,size,n", [([7], [300], 3), ([3, 2], [19, 33], 2), ([2, 1, 2], [9, 11, 10], 2)])
def test_kept_A_matches_the_calls_that_make_it_twice(cuda, nc, size, n):
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=True)
    p, L = T.params, N.lib()
    gen = torch.Generator().manual_seed(3)
    theta = (torch.randn(n, p.d, generator=gen) * 0.2).to(cuda).requires_grad_(True)
    data = torch.rand([n, 2] + size, generator=gen).to(cuda)
    pts = torch.rand(len(nc), 500, generator=gen).to(cuda)
    dev = H.device_tess(p, theta.device)
    st = H._stream(theta.device)

    out = T.transform_data(data, theta, size)
    up = torch.rand(out.shape, generator=gen).to(cuda)
    got, = torch.autograd.grad(out, theta, up)
    lin, sz, nP = H.meshgrid_axes(size, cuda), H._int_arr(size), out[0, 0].numel()
    ws, nb = dev.workspace(n, nP, size)
    saved = torch.empty(L.cpab_saved_floats(len(nc), n, nP), device=cuda)
    out2, want = torch.empty_like(out), torch.empty_like(theta)
    N.check(L.cpab_transform_data_fwd(dev.ref, theta.data_ptr(), n, data.data_ptr(), 2, sz, sz, lin.data_ptr(), 1.0,
                                      out2.data_ptr(), saved.data_ptr(), ws.data_ptr(), nb, st))
    N.check(L.cpab_transform_data_bwd(dev.ref, theta.data_ptr(), n, data.data_ptr(), 2, sz, sz, lin.data_ptr(), 1.0,
                                      up.data_ptr(), saved.data_ptr(), None, want.data_ptr(), ws.data_ptr(), nb, st))
    assert torch.equal(out, out2) and torch.equal(got, want)

    out = T.transform_grid(pts, theta)
    up = torch.rand(out.shape, generator=gen).to(cuda)
    got, = torch.autograd.grad(out, theta, up)
    ws, nb = dev.workspace(n, 500)
    jac = torch.empty(L.cpab_jac_floats(len(nc), n, 500), device=cuda)
    out2 = torch.empty_like(out)
    N.check(L.cpab_transform_fwd(dev.ref, theta.data_ptr(), n, pts.data_ptr(), 500, 0, None, 1.0, out2.data_ptr(),
                                 jac.data_ptr(), ws.data_ptr(), nb, st))
    N.check(L.cpab_transform_bwd(dev.ref, theta.data_ptr(), n, pts.data_ptr(), 500, 0, None, 1.0, up.data_ptr(),
                                 jac.data_ptr(), want.data_ptr(), None, ws.data_ptr(), nb, st))
    assert torch.equal(out, out2) and torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("nc,zb", [([2], True), ([40], True), ([3, 3], True), ([2, 3], False), ([1, 2, 1], True),
                                   ([1, 1, 1], False)])
@pytest.mark.parametrize("n,nP", [(1, 1), (2, 300), (1, 65536), (1, 65537), (257, 20)])
def test_the_forward_that_makes_A_leaves_the_same_bits(cuda, nc, zb, n, nP):
    """Up to 256 blocks the forward makes A itself; cpab_theta_to_A is always a launch of its own."""
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=zb)
    L, dev = N.lib(), H.device_tess(T.params, cuda)
    gen = torch.Generator().manual_seed(4)
    theta = (torch.randn(n, T.params.d, generator=gen) * 0.2).to(cuda)
    pts = (torch.rand(len(nc), nP, generator=gen) * 1.2 - 0.1).to(cuda)
    A, want = dev.new_A(theta).fill_(float("nan")), dev.new_A(theta)
    st, out = H._stream(theta.device), torch.empty(n, len(nc), nP, device=cuda)
    N.check(L.cpab_transform_fwd_keep(dev.ref, theta.data_ptr(), n, pts.data_ptr(), nP, 0, None, 1.0, out.data_ptr(),
                                      None, A.data_ptr(), 4 * A.numel(), st))
    N.check(L.cpab_theta_to_A(dev.ref, theta.data_ptr(), n, want.data_ptr(), st))
    assert torch.equal(A, want) and torch.isfinite(out).all()


def test_kept_A_argument_errors():
    L, t = N.lib(), N.CpabTess()
    t.ndim, t.nc, t.nC, t.d, t.planes, t.nbr, t.B = 2, N.int3([2, 2]), 16, 10, 1, 1, 1
    need = 3 * 16 * 6 * 4
    sz = (ctypes.c_int * 3)(8, 8, 1)
    # (no GPU work is started: every call returns before a launch)
    assert L.cpab_transform_fwd_keep(ctypes.byref(t), 1, 3, 1, 10, 0, None, 1.0, 1, None, 1, need - 1, None) == 3
    assert L.cpab_transform_fwd_keep(ctypes.byref(t), 1, 3, 1, 10, 0, None, 1.0, 1, None, None, need, None) == 3
    assert L.cpab_transform_bwd_kept(ctypes.byref(t), None, 3, 1, 10, 0, None, 1.0, 1, None, 1, None, 1, 1 << 20,
                                     None) == 1
    assert L.cpab_transform_bwd_kept(ctypes.byref(t), 1, 3, 1, 10, 0, None, 1.0, 1, None, 1, None, 1, 8, None) == 3
    assert L.cpab_transform_data_fwd_keep(ctypes.byref(t), 1, 3, 1, 1, sz, sz, 1, 1.0, 1, None, 1, need - 1, None) == 3
    assert L.cpab_transform_data_bwd_kept(ctypes.byref(t), None, 3, 1, 1, sz, sz, 1, 1.0, 1, None, None, 1, 1, 1 << 20,
                                          None) == 1
    assert L.cpab_transform_data_bwd_kept(ctypes.byref(t), 1, 3, 1, 1, sz, sz, 1, 1.0, 1, None, None, 1, 1, 8, None) == 3
