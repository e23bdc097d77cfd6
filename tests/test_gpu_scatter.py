"""dL/ddata of the interpolation (cpab_interpolate_bwd): lanes of a wave hand
the weights of their upper samples to the neighbouring lane whose lower samples
they are, and only the rest goes to memory.  Every way that can go wrong against
the FP64 restatement: rows that end inside a wave, waves that span two
instances, neighbours that do not line up (stretched, folded and random grids),
points beyond the first and last sample, up- and down-sampling."""
import numpy as np
import pytest
import torch

import oracle as O
from libcpab_amd import _native as N
from libcpab_amd.pytorch import hip_ops as H

pytestmark = pytest.mark.gpu


def _grid(kind, n, out, rng):
    nd = len(out)
    mesh = O.uniform_meshgrid(out)
    if kind == "random":
        return rng.uniform(-0.1, 1.1, (n,) + mesh.shape)
    x = np.repeat(mesh[None], n, 0)
    if kind == "stretched":
        return 1.2 * x - 0.1
    if kind == "folded":  # runs backwards past the middle
        return 1.0 - np.abs(1.0 - 1.7 * x)
    shift = 0.03 * np.sin(6.0 * x[:, ::-1] + rng.uniform(0, 6, (n, nd, 1)))
    return x + (shift if kind == "warped" else 0.0)


@pytest.mark.parametrize("kind", ["identity", "warped", "stretched", "folded", "random"])
@pytest.mark.parametrize("size,out,n,c", [((65,), (65,), 3, 2), ((40,), (131,), 2, 1), ((300,), (63,), 5, 1),
                                          ((33, 17), (33, 17), 2, 3), ((16, 16), (16, 16), 1, 5),
                                          ((20, 9), (50, 31), 2, 1), ((64, 70), (20, 7), 1, 2), ((1, 12), (9, 12), 2, 1),
                                          ((9, 10, 11), (9, 10, 11), 2, 2), ((5, 6, 4), (11, 13, 9), 3, 1),
                                          ((20, 2, 18), (7, 9, 8), 1, 1)])
def test_data_gradient_of_merged_lanes(cuda, size, out, n, c, kind):
    rng = np.random.default_rng(5)
    nd = len(size)
    grid = _grid(kind, n, list(out), rng).astype(np.float32)
    data = rng.standard_normal((n, c) + size).astype(np.float32)
    g = rng.standard_normal((n, c) + out).astype(np.float32)
    want, _ = O.interpolate_backward(nd, data, grid, list(out), g, index32=True)
    size_of_terms, _ = O.interpolate_backward(nd, data, grid, list(out), np.abs(g), index32=True)
    t = [torch.tensor(a, device=cuda) for a in (data, grid, g)]
    got = torch.zeros_like(t[0])
    N.check(N.lib().cpab_interpolate_bwd(nd, H._ptr(t[0]), n, c, H._int_arr(size), H._ptr(t[1]), H._int_arr(out),
                                         H._ptr(t[2]), H._ptr(got), None, H._stream(got.device)))
    # every term's weight is off by a few eps (absolute), every addition by eps of the partial sum
    tol = 64 * 2.0 ** -24 * (np.abs(size_of_terms) + 8 * np.abs(g).max())
    assert (np.abs(got.cpu().double().numpy() - want) <= tol).all()


@pytest.mark.parametrize("nc,size,out,c", [([3, 3], (31, 20), (31, 20), 5), ([2, 2, 2], (10, 12, 9), (10, 12, 9), 2),
                                           ([2, 2, 2], (6, 20, 5), (9, 17, 3), 1), ([12], (150,), (150,), 3)])
def test_fused_data_gradient_equals_the_interpolation_of_the_warped_grid(cuda, nc, size, out, c):
    from libcpab_amd import Cpab
    T = Cpab(nc, backend="pytorch", device="gpu")
    gen = torch.Generator().manual_seed(3)
    n = 3
    theta = (torch.randn(n, T.get_theta_dim(), generator=gen) * 0.3).to(cuda)
    data = torch.randn((n, c) + size, generator=gen).to(cuda).requires_grad_(True)
    g = torch.randn((n, c) + out, generator=gen)
    (got,) = torch.autograd.grad(T.transform_data(data, theta, list(out)), data, g.to(cuda))
    warped = T.transform_grid(T.uniform_meshgrid(list(out)), theta).cpu().numpy()
    nd = len(nc)
    want, _ = O.interpolate_backward(nd, data.detach().cpu().numpy(), warped, list(out), g.numpy(), index32=True)
    terms, _ = O.interpolate_backward(nd, data.detach().cpu().numpy(), warped, list(out), g.abs().numpy(), index32=True)
    # the two routes' points may differ by one ulp: a weight by size * 2^-24
    tol = 64 * 2.0 ** -24 * (np.abs(terms) + 8 * g.abs().max().item()) + 8 * max(size) * 2.0 ** -23 * g.abs().max().item()
    assert (np.abs(got.cpu().double().numpy() - want) <= tol).all()
