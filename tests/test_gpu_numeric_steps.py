"""method='numeric': the cell lookup's FP32 path against the reference's rules
where it must give way to them, and dL/dtheta as the adjoint of the steps
against the products of the per-theta derivatives it replaces."""
import numpy as np
import pytest
import torch

import oracle as O
from libcpab_amd import Cpab
from libcpab_amd import _native as N
from libcpab_amd.pytorch import hip_ops as H

pytestmark = pytest.mark.gpu


def _near_facets(nc, rng, n=4000):
    """Points whose scaled coordinates sit on grid lines, diagonals and planes
    through cell corners, moved by up to a few ulps or up to 1e-4, some outside."""
    nd = len(nc)
    q = rng.uniform(-0.3, 1.3, (nd, n)) * np.array(nc)[:, None]
    line = rng.integers(0, 3, (nd, n))
    q = np.where(line == 0, np.round(q), q)
    if nd > 1:  # u = v, u = 1 - v, and in 3D u + v + w = 1 or 2 in local coordinates
        base = np.floor(q)
        u = q - base
        k = rng.integers(0, 4, n)
        u[1] = np.where(k == 1, u[0], np.where(k == 2, 1 - u[0], u[1]))
        if nd == 3:
            u[2] = np.where(k == 3, np.abs(1 - u[0] - u[1]), u[2])
        q = base + u
    x = (q / np.array(nc)[:, None]).astype(np.float32)
    ulps = rng.integers(-3, 4, (nd, n)).astype(np.float32) * np.spacing(np.abs(x).astype(np.float32))
    far = rng.uniform(-1e-4, 1e-4, (nd, n)) * (rng.random((nd, n)) < 0.3)
    return np.ascontiguousarray(x + ulps + far.astype(np.float32))


@pytest.mark.parametrize("nc", [[7], [3, 2], [8, 8], [1, 5], [2, 3, 2], [3, 1, 2], [1, 1, 4]])
def test_steps_near_facets_are_bit_exact(cuda, nc):
    rng = np.random.default_rng(1)
    nd = len(nc)
    pts = _near_facets(nc, rng)
    A = rng.standard_normal((2, O.n_cells(nd, nc), nd, nd + 1)) * 0.5
    trels = O.trels(A, 20).astype(np.float32)
    want = O.step_forward_f32(nd, nc, 3, pts, trels)
    t = [torch.tensor(a, device=cuda) for a in (pts, trels)]
    out = torch.empty(2, nd, pts.shape[1], device=cuda)
    N.check(N.lib().cpab_ref_forward(H._ptr(out), H._ptr(t[0]), H._ptr(t[1]), 3, H._int_arr(nc), nd, pts.shape[1], 2, 0,
                                     H._stream(out.device)))
    assert np.array_equal(out.cpu().numpy(), want, equal_nan=True)


@pytest.mark.parametrize("nc", [[9], [3, 2], [2, 1, 3]])
@pytest.mark.parametrize("n,points,steps,cloud", [(1, 1, 1, False), (3, 63, 2, False), (2, 64, 7, True),
                                                  (2, 65, 50, False), (1, 1500, 121, False), (4, 300, 16, True)])
def test_gradient_is_the_sum_of_the_derivatives(cuda, nc, n, points, steps, cloud):
    from libcpab_amd import Cpab
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=len(nc) != 2)
    T.set_solver_params(nstepsolver=steps, method="numeric")
    p, nd = T.get_params(), len(nc)
    gen = torch.Generator().manual_seed(4)
    theta = (torch.randn(n, p.d, generator=gen) * 0.4).to(cuda).requires_grad_(True)
    shape = (n, nd, points) if cloud else (nd, points)
    pts = (torch.rand(shape, generator=gen) * 1.1 - 0.05).to(cuda)
    g = torch.randn(n, nd, points, generator=gen).to(cuda)
    (got,) = torch.autograd.grad(T.transform_grid(pts, theta), theta, g)
    dev = H.device_tess(p, theta.device)
    As = (dev.B @ theta.detach().t()).t().contiguous()
    Bs = dev.B.t().contiguous()
    J = torch.empty(p.d, n, nd, points, device=cuda)
    N.check(N.lib().cpab_ref_backward(H._ptr(J), H._ptr(pts), H._ptr(As), H._ptr(Bs), steps, H._int_arr(nc), n, p.d, nd,
                                      points, p.nC, int(cloud), H._stream(J.device)))
    terms = J.double() * g.double()
    want = terms.sum((2, 3)).t()
    # a derivative takes `steps` roundings, the sums a few more
    tol = (8 * steps + 64) * 2.0 ** -24 * terms.abs().sum((2, 3)).max()
    assert (got.double() - want).abs().max() <= tol


def test_more_steps_than_the_lds_holds_take_the_derivatives(cuda):
    """2 sqrt(steps) points per lane of a 64-lane block beside the tables of 400
    cells: past the LDS the workspace size is 0 and every derivative is formed."""
    from libcpab_amd import Cpab
    T = Cpab([10, 10], backend="pytorch", device="gpu")
    p = T.get_params()
    assert N.lib().cpab_ref_grad_workspace_bytes(2, H._int_arr([10, 10]), 1, 40, 50) > 0
    assert N.lib().cpab_ref_grad_workspace_bytes(2, H._int_arr([10, 10]), 1, 40, 40000) == 0
    gen = torch.Generator().manual_seed(4)
    theta = (torch.randn(1, p.d, generator=gen) * 0.1).to(cuda).requires_grad_(True)
    pts = torch.rand(2, 40, generator=gen).to(cuda)
    g = torch.ones(1, 2, 40, device=cuda)
    grads = []
    for steps in (50, 40000):
        T.set_solver_params(nstepsolver=steps, method="numeric")
        grads.append(torch.autograd.grad(T.transform_grid(pts, theta), theta, g)[0])
    # the scheme's own error at 50 steps is O(1 / steps^2); FP32 rounding over 40000
    assert (grads[0] - grads[1]).abs().max() <= 2e-2 * grads[0].abs().max()


@pytest.mark.parametrize("nc,n", [([2], 1), ([40], 3), ([3, 3], 2), ([1, 1, 1], 2), ([2, 2, 3], 2)])
def test_expanded_parameters_and_their_exponentials(cuda, nc, n):
    """A = B theta and expm(A~ / nstep) of every cell, at cell counts around a block's 32, against FP64: A within the
    rounding of its d products, the exponential within half an FP32 unit of that of the A returned."""
    T = Cpab(nc, backend="pytorch", device="gpu", zero_boundary=len(nc) < 3)
    dev = H.device_tess(T.params, cuda)
    ndim, nC, d = len(nc), T.params.nC, T.get_theta_dim()
    theta = torch.randn(n, d, generator=torch.Generator().manual_seed(1)).to(cuda)
    As = torch.empty(n, nC, ndim, ndim + 1, device=cuda)
    trels = torch.empty_like(As)
    N.check(N.lib().cpab_ref_expand(dev.ref, H._ptr(theta), n, 50, H._ptr(As), H._ptr(trels), H._stream(theta.device)))
    B, th = dev.B.double(), theta.double()
    want = th.cpu() @ B.t().cpu()
    size = th.abs().cpu() @ B.t().abs().cpu()
    assert ((As.double().cpu().reshape(n, -1) - want).abs() <= (d + 1) * 2.0 ** -24 * size + 1e-30).all()
    X = torch.zeros(n, nC, ndim + 1, ndim + 1, dtype=torch.float64)
    X[:, :, :ndim] = As.double().cpu() / 50
    E = torch.linalg.matrix_exp(X)[:, :, :ndim]
    assert ((trels.double().cpu() - E).abs() <= 1.01 * 2.0 ** -24 * E.abs() + 2e-9 * X.abs().amax()).all()
