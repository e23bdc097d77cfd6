"""The steps of the 1D gradient's pass, compiled for the host: they are the
forward's bit for bit, with and without the table of whole-cell crossings, and
phi1 and phi2 are no further from 64 bits than the library's quotients."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

import oracle as O
from conftest import ROOT
from libcpab_amd.core.tessellation import make_tessellation

SRC = os.path.join(ROOT, "tests", "host_signal.cpp")
OUT = os.path.join(ROOT, "tests", "_build", "libhostsignal.so")


def _lib():
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    deps = [SRC, os.path.join(ROOT, "libcpab_amd", "csrc", "cpab_device.hpp")]
    if not os.path.exists(OUT) or os.path.getmtime(OUT) < max(os.path.getmtime(d) for d in deps):
        if not os.path.exists(hipcc):
            pytest.skip("hipcc not available")
        os.makedirs(os.path.dirname(OUT), exist_ok=True)
        tmp = "%s.%d" % (OUT, os.getpid())
        subprocess.check_call([hipcc, "-x", "hip", "--offload-host-only", "-O2", "-fPIC", "-shared", "-o", tmp, SRC])
        os.replace(tmp, OUT)
    return ctypes.CDLL(OUT)


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


@pytest.mark.parametrize("which", [0, 1, 2], ids=["gradient", "table", "gradient_table"])
@pytest.mark.parametrize("nc", [1, 2, 7, 50, 200])
@pytest.mark.parametrize("free", [False, True])
@pytest.mark.parametrize("scale", [1e-4, 0.5, 3.0])
def test_every_pass_takes_the_same_steps(nc, free, scale, which):
    if nc == 1 and not free:
        pytest.skip("one cell with a fixed point at each end has no field")
    T = make_tessellation([nc], zero_boundary=not free)
    rng = np.random.default_rng(11)
    theta = rng.standard_normal((4, T.B.shape[1])) * scale
    Aq = O.expand_A(T.B, theta, 1).reshape(4, nc, 2).astype(np.float32)
    Aq[..., 1] *= nc
    x = np.concatenate([np.linspace(0, 1, 4 * nc + 1), rng.uniform(0, 1, 3000)]).astype(np.float32)
    for A in Aq:
        assert _lib().host_signal_mismatches(nc, _ptr(np.ascontiguousarray(A)), _ptr(x), x.size, which) == 0


def test_phis_against_64_bits():
    z = np.concatenate([s * np.geomspace(1e-6, 20, 200001) for s in (-1, 1)]).astype(np.float32)
    p1, p2 = np.zeros_like(z), np.zeros_like(z)
    _lib().host_phis(_ptr(z), z.size, _ptr(p1), _ptr(p2))
    w = z.astype(np.longdouble)
    e1 = np.expm1(w) / w
    # phi2 as a sum where the difference cancels
    s, t = np.full_like(w, 0.5), np.full_like(w, 0.5)
    for k in range(3, 40):
        t = t * w / k
        s = s + t
    e2 = np.where(np.abs(w) < 2, s, (np.expm1(w) - w) / w ** 2)
    # the sum: its last step's rounding, and |z| times the one before (|z| <= 1, the
    # results are above 0.26); the quotients: one for expm1 (an ulp), one each for the
    # difference, the square and the quotient, expm1's against a difference of at
    # least 1 / 2.4 of it
    u = 2.0 ** -24
    small = np.abs(z) <= 1
    r1, r2 = np.abs(p1 / e1 - 1), np.abs(p2 / e2 - 1)
    assert r1[small].max() <= 2 * u and r2[small].max() <= 2 * u
    assert r1[~small].max() <= 3 * u and r2[~small].max() <= (2.4 * 2 + 3) * u
