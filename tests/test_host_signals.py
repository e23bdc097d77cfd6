"""The 1D closed form compiled for the host: fields strong enough to leave the
range of its Taylor sums (|a| h > 1), cells entered at their edges, fixed points
inside cells and at edges, against the FP64 flow."""
import numpy as np
import pytest

import oracle as O
from libcpab_amd.core.tessellation import make_tessellation
from test_host_integrator import host_transform


@pytest.mark.parametrize("nc", [[1], [2], [7], [64]])
@pytest.mark.parametrize("free", [False, True])
@pytest.mark.parametrize("scale", [1e-4, 0.5, 3.0])
def test_signal_flow_over_weak_and_strong_fields(nc, free, scale):
    if nc == [1] and not free:
        pytest.skip("one cell with a fixed point at each end has no field")
    T = make_tessellation(nc, zero_boundary=not free)
    planes, nbr = T.facet_table()
    rng = np.random.default_rng(7)
    theta = rng.standard_normal((4, T.B.shape[1])) * scale
    x = np.concatenate([np.linspace(0, 1, 16 * nc[0] + 1), rng.uniform(0, 1, 300)])[None].astype(np.float32)
    out, jac = host_transform(nc, T.B, planes, nbr, theta, x, want_jac=True)
    want = O.cf_forward(1, nc, O.expand_A(T.B, theta, 1), planes, nbr, x.astype(np.float64))
    # FP32 A and positions (nc-scaled, eps/2 each) carried by the flow: a handful of
    # roundings per cell passed, grown by at most the largest stretch met
    stretch = 1 + np.abs(jac).max(axis=(1, 2), keepdims=True)
    passed = 4 + np.abs(out - x).max() * nc[0]
    tol = 4 * passed * 2.0 ** -24 * stretch * (1 + np.abs(want))
    assert (np.abs(out - want) <= tol).all()
