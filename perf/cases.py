"""Performance cases: the calls a program makes of this framework, over the sizes it makes them at.

A case is a dict of plain values; ``prepare`` makes what the program has in hand (transformer, parameters, data,
upstream gradient) on the GPU, ``run`` is one pass through the public entry points, ``exact`` the same outputs in 64
bits by plain torch.

Kinds of call
    grid      Cpab.transform_grid on explicit points (shared, or a cloud for each theta)
    data      Cpab.transform_data: meshgrid, integration, interpolation
    chain     CpabSequential.transform_data
    ragged    CpabBatch: many problems of different sizes in one captured launch sequence
    numeric   Cpab.transform_grid with method='numeric', the fixed-step scheme

Images, volumes and signals are smooth, and so are the upstream gradients, as those of two registered acquisitions
are.  That also makes dL/dtheta a well-posed number: linear interpolation has another slope on each side of a sample,
so between noisy samples a point that rounds to the other side changes the sum in any precision.
"""
import math
import random

import torch

from libcpab_amd import Cpab, CpabSequential
from libcpab_amd.batch import CpabBatch

F64 = torch.float64


def listed():
    return [
        # the deformation of one picture's grid, to look at or to resample with: the smallest call, all latency
        dict(name="grid_one_2d", kind="grid", tess="3x3", free=False, n=1, points=10000, cloud=False, mesh=True,
             grad="", scale=0.3),
        # one step of registering a pair of pictures by gradient descent on theta
        dict(name="pair_2d", kind="data", tess="4x4", free=False, n=1, channels=3, size="256x256", out="256x256",
             grad="theta", scale=0.3),
        # a transformer layer on small feature maps inside a network: both gradients, small images, many of them
        dict(name="layer_2d", kind="data", tess="3x3", free=False, n=128, channels=1, size="64x64", out="64x64",
             grad="theta+data", scale=0.3),
        # the image workload of bench.py: a large training batch
        dict(name="images_2d", kind="data", tess="4x4", free=False, n=256, channels=3, size="256x256", out="256x256",
             grad="theta+data", scale=0.3),
        # augmentation: forward only, free boundary, odd sizes, another output size than the input's
        dict(name="augment_2d", kind="data", tess="6x5", free=True, n=48, channels=3, size="301x211", out="223x224",
             grad="", scale=0.1),
        # the time-series workload of bench.py: aligning many signals
        dict(name="signals_1d", kind="data", tess="50", free=False, n=4096, channels=1, size="1024", out="1024",
             grad="theta", scale=0.5),
        # the volume workload of bench.py: registering volumes
        dict(name="volumes_3d", kind="data", tess="3x3x3", free=False, n=16, channels=1, size="64x64x64",
             out="64x64x64", grad="theta", scale=0.2),
        # a volumetric layer inside a network: both gradients, ragged sizes
        dict(name="layer_3d", kind="data", tess="2x2x2", free=False, n=6, channels=2, size="49x40x35", out="49x40x35",
             grad="theta+data", scale=0.2),
        # landmarks or surface points, another cloud for each theta, both gradients
        dict(name="clouds_3d", kind="grid", tess="2x2x2", free=False, n=16, points=25001, cloud=True, mesh=False,
             grad="theta+points", scale=0.2),
        # the composition workload of bench.py: four transforms in a row, trained together
        dict(name="chain_2d", kind="chain", tess="4x4", free=False, stages=4, n=64, channels=3, size="256x256",
             out="256x256", grad="theta", scale=0.3),
        # a mixed batch of signals and pictures, each of its own size and tessellation
        dict(name="ragged", kind="ragged", instances=200, mix=1, scale=0.3),
        # the fixed-step integrator and its gradient, for results comparable step by step with published ones
        dict(name="numeric_2d", kind="numeric", tess="3x3", free=False, n=8, points=10000, steps=50, grad="theta",
             scale=0.3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _text(v):
    return "x".join(str(int(x)) for x in v)


def draw(rng):
    kind = rng.choice(["data1", "data2", "data2", "data3", "grid", "chain", "ragged", "numeric"])
    grad = rng.choice(["", "theta", "theta+data", "theta+data"])
    if kind == "data1":
        size = _log_int(rng, 200, 8192)
        n = max(1, min(4096, _log_int(rng, 1, 4.0e6 / size)))
        return dict(kind="data", tess=str(rng.randint(10, 100)), free=False, n=n, channels=rng.choice([1, 1, 2, 3]),
                    size=str(size), out=str(size if rng.random() < 0.6 else _log_int(rng, size / 2, size)), grad=grad,
                    scale=round(rng.uniform(0.2, 0.5), 3))
    if kind == "data2":
        size = [_log_int(rng, 64, 512), _log_int(rng, 64, 512)]
        out = size if rng.random() < 0.6 else [max(64, int(s * rng.uniform(0.6, 1.0))) for s in size]
        n = max(1, min(256, _log_int(rng, 1, 1.0e7 / (size[0] * size[1]))))
        free = rng.random() < 0.2
        return dict(kind="data", tess=_text([rng.randint(2, 8), rng.randint(2, 8)]), free=free, n=n,
                    channels=rng.choice([1, 3, 3, 4]), size=_text(size), out=_text(out), grad="" if free else grad,
                    scale=0.1 if free else round(rng.uniform(0.1, 0.3), 3))
    if kind == "data3":
        size = [_log_int(rng, 24, 96) for _ in range(3)]
        n = max(1, min(16, _log_int(rng, 1, 3.0e6 / (size[0] * size[1] * size[2]))))
        return dict(kind="data", tess=_text([rng.randint(1, 3) for _ in range(3)]), free=False, n=n,
                    channels=rng.choice([1, 1, 2]), size=_text(size), out=_text(size), grad=grad,
                    scale=round(rng.uniform(0.1, 0.2), 3))
    if kind == "grid":
        nd = rng.choice([2, 3])
        points = _log_int(rng, 1000, 100000)
        n = max(1, min(64, _log_int(rng, 1, 1.0e6 / points)))
        return dict(kind="grid", tess=_text([rng.randint(2, 4) for _ in range(2)] if nd == 2 else [2, rng.randint(1, 3), 2]),
                    free=False, n=n, points=points, cloud=rng.random() < 0.5, mesh=False,
                    grad=rng.choice(["", "theta", "theta+points"]), scale=round(rng.uniform(0.1, 0.3), 3))
    if kind == "chain":
        size = [_log_int(rng, 96, 256), _log_int(rng, 96, 256)]
        return dict(kind="chain", tess=_text([rng.randint(2, 5), rng.randint(2, 5)]), free=False,
                    stages=rng.randint(2, 4), n=_log_int(rng, 2, 48), channels=rng.choice([1, 3]), size=_text(size),
                    out=_text(size), grad="theta", scale=round(rng.uniform(0.1, 0.3), 3))
    if kind == "ragged":
        return dict(kind="ragged", instances=rng.randint(20, 160), mix=rng.randint(2, 10 ** 6), scale=0.3)
    return dict(kind="numeric", tess=_text([rng.randint(2, 3), rng.randint(2, 3)]), free=False, n=rng.randint(1, 6),
                points=_log_int(rng, 1000, 10000), steps=rng.choice([20, 50]), grad=rng.choice(["", "theta", "theta"]),
                scale=round(rng.uniform(0.1, 0.3), 3))


# ----------------------------------------------------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------------------------------------------------
def _ints(text):
    return [int(v) for v in text.split("x")]


def _smooth(gen, lead, size):
    """[*lead, *size] float32: for each leading entry a shading of at most 0.4 cycles along each axis."""
    dev, nd = gen.device, len(size)
    n = math.prod(lead)
    freq = torch.rand(n, nd, generator=gen, device=dev) * 0.3 + 0.1
    arg = 6.2831853 * torch.rand(n, generator=gen, device=dev).reshape((n,) + (1,) * nd)
    for a, s in enumerate(size):
        shape = [1] * (nd + 1)
        shape[a + 1] = s
        arg = arg + 6.2831853 * freq[:, a].reshape((n,) + (1,) * nd) * torch.linspace(0, 1, s, device=dev).reshape(shape)
    return (0.5 + 0.4 * torch.cos(arg)).reshape(tuple(lead) + tuple(size)).contiguous()


def _problems(case):
    """(tessellation, channels, size) of each instance of a ragged mix: half signals (10-100 cells, 256-8192 points),
    half pictures (2-8 cells and 64-512 pixels along an axis, 3 channels)."""
    rng, out = random.Random(case["mix"]), []
    for _ in range(case["instances"]):
        if rng.random() < 0.5:
            out.append(([rng.randint(10, 100)], 1, [_log_int(rng, 256, 8192)]))
        else:
            s = _log_int(rng, 64, 512)
            out.append(([rng.randint(2, 8), rng.randint(2, 8)], 3, [s, s]))
    return out


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "ragged":
        probs, made = [], {}
        for nc, channels, size in _problems(case):
            T = made.setdefault(tuple(nc), None) or Cpab(nc, backend="pytorch", device="gpu", zero_boundary=True)
            made[tuple(nc)] = T
            probs.append((T, channels, size, size))
        b = CpabBatch(probs, device="cuda", save=True)
        for i, (T, channels, size, _) in enumerate(probs):
            b.theta_views[i].copy_(torch.randn(T.get_theta_dim(), generator=gen, device="cuda") * case["scale"])
            b.data_views[i].copy_(_smooth(gen, (channels,), size))
            b.grad_out_views[i].copy_(_smooth(gen, (channels,), size))
        b.capture()
        return dict(kind=kind, batch=b, probs=probs)
    nc = _ints(case["tess"])
    Ts = [Cpab(nc, backend="pytorch", device="gpu", zero_boundary=not case["free"])
          for _ in range(case.get("stages", 1))]
    n, d, nd = case["n"], Ts[0].get_theta_dim(), len(nc)
    wants = case["grad"].split("+")
    thetas = [(torch.randn(n, d, generator=gen, device="cuda") * case["scale"]).requires_grad_("theta" in wants)
              for _ in Ts]
    s = dict(kind=kind, T=Ts[0], thetas=thetas, wrt=list(thetas) if "theta" in wants else [])
    if kind in ("data", "chain"):
        size, s["out"] = _ints(case["size"]), _ints(case["out"])
        s["data"] = _smooth(gen, (n, case["channels"]), size).requires_grad_("data" in wants)
        s["upstream"] = _smooth(gen, (n, case["channels"]), s["out"])
        s["wrt"] += [s["data"]] if "data" in wants else []
        s["chain"] = CpabSequential(*Ts) if kind == "chain" else None
        return s
    if kind == "numeric":
        Ts[0].set_solver_params(nstepsolver=case["steps"], method="numeric")
    points = case["points"]
    if case.get("mesh"):
        side = int(round(math.sqrt(points)))
        s["grid"] = Ts[0].uniform_meshgrid([side, side])
    else:
        shape = (n, nd, points) if case.get("cloud") else (nd, points)
        s["grid"] = torch.rand(shape, generator=gen, device="cuda").requires_grad_("points" in wants)
    s["wrt"] += [s["grid"]] if "points" in wants else []
    # the upstream gradient of a distance to targets that lie one way from the points
    s["upstream"] = torch.rand(n, nd, s["grid"].shape[-1], generator=gen, device="cuda") + 0.2
    return s


def run(s):
    if s["kind"] == "ragged":
        b = s["batch"]
        b.replay_forward()
        b.replay_backward()
        return {"out": b.out, "grad_theta": b.grad_theta, "grad_data": b.grad_data}
    if s["kind"] == "data":
        out = s["T"].transform_data(s["data"], s["thetas"][0], s["out"])
    elif s["kind"] == "chain":
        out = s["chain"].transform_data(s["data"], s["thetas"], s["out"])
    else:
        out = s["T"].transform_grid(s["grid"], s["thetas"][0])
    if not s["wrt"]:
        return [out]
    return [out.detach()] + list(torch.autograd.grad(out, s["wrt"], s["upstream"]))


# ----------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------------------------------------------------
# operations per point of one flow: velocity, series and one facet search (forward), adjoint and the integral (backward)
_FWD = {1: 20, 2: 120, 3: 250}
_BWD = {1: 40, 2: 240, 3: 600}


def _work_data(nd, n, channels, size, out, grad, stages, d):
    p, m = n * math.prod(out), n * math.prod(size)
    values = m * channels + p * channels + stages * n * d
    flops = p * (stages * _FWD[nd] + channels * 3 * 2 ** nd)
    if grad:
        values += p * channels + m * channels + stages * n * d  # upstream and data again, dL/dtheta
        flops += p * (stages * _BWD[nd] + channels * 6 * 2 ** nd)
        values += m * channels if "data" in grad else 0
    return values * 4, flops


def work(case):
    kind = case["kind"]
    if kind == "ragged":
        got = [_work_data(len(nc), 1, c, size, size, "theta+data", 1, 0) for nc, c, size in _problems(case)]
        return {"bytes": sum(b for b, _ in got), "flops": sum(f for _, f in got)}
    nc = _ints(case["tess"])
    nd, n, grad = len(nc), case["n"], case["grad"]
    if kind in ("data", "chain"):
        b, f = _work_data(nd, n, case["channels"], _ints(case["size"]), _ints(case["out"]), grad,
                          case.get("stages", 1), 2 * math.prod(nc))
        return {"bytes": b, "flops": f}
    p = case["points"]
    clouds = n if case.get("cloud") else 1
    values = nd * p * (clouds + n)
    flops = n * p * (_FWD[nd] if kind == "grid" else case["steps"] * 2 * nd * nd)
    if grad:
        values += nd * p * (clouds + n) + (nd * p * clouds if "points" in grad else 0)
        # numeric: a midpoint step of the point and of its derivative along each theta entry (at least two a cell)
        flops += n * p * (_BWD[nd] if kind == "grid" else case["steps"] * 8 * nd * nd * 2 * math.prod(nc))
    return {"bytes": 4 * values, "flops": flops}


# ----------------------------------------------------------------------------------------------------------------------
# the same outputs in 64 bits
# ----------------------------------------------------------------------------------------------------------------------
def _cells(x, nc):
    """Cell of each point x [N, D] under nc [N, D]: the tessellation's definition."""
    D = x.shape[1]
    q = x * nc
    if D == 3:  # inside the domain (a point on a face is kept inside)
        q = torch.minimum(q.clamp(min=0), nc)
    base = torch.minimum(q.floor().clamp(min=0), nc - 1)
    if D == 1:
        return base[:, 0].long()
    u = q - base
    if D == 2:
        a, b = u[:, 0] < u[:, 1], 1 - u[:, 0] < u[:, 1]
        tri = torch.where(a, torch.where(b, 2, 3), torch.where(b, 1, 0))
        x0, x1 = x[:, 0], x[:, 1]
        # beyond an edge and beside the corners' diagonals the edge's own triangle reaches out
        lo0, hi0, lo1, hi1 = x0 <= 0, x0 >= 1, x1 <= 0, x1 >= 1
        tri = torch.where(hi1 & ~lo0 & ~hi0, 2, tri)
        tri = torch.where(lo1 & ~lo0 & ~hi0, 0, tri)
        tri = torch.where(hi0 & ~lo1 & ~hi1, 1, tri)
        tri = torch.where(lo0 & ~lo1 & ~hi1, 3, tri)
        return (4 * (base[:, 0] + base[:, 1] * nc[:, 0])).long() + tri
    odd = (base.sum(1) % 2) == 1
    a, b, c = torch.where(odd, u[:, 1], u[:, 0]), torch.where(odd, 1 - u[:, 0], u[:, 1]), u[:, 2]
    tet = torch.where(-a - b + c >= 0, 1, torch.where(a + b + c - 2 >= 0, 2, torch.where(
        -a + b - c >= 0, 3, torch.where(a - b - c >= 0, 4, 0))))
    return (5 * (base[:, 0] + base[:, 1] * nc[:, 0] + base[:, 2] * nc[:, 0] * nc[:, 1])).long() + tet


_INNER = {1: [[0.5]], 2: [[1 / 2, 1 / 6], [5 / 6, 1 / 2], [1 / 2, 5 / 6], [1 / 6, 1 / 2]],
          3: [[0.5, 0.5, 0.5], [0.25, 0.25, 0.75], [0.75, 0.75, 0.75], [0.25, 0.75, 0.25], [0.75, 0.25, 0.25]]}


def _inner(cell, nc):
    """A point inside each cell."""
    D = nc.shape[1]
    table = torch.tensor(_INNER[D], dtype=F64, device=nc.device)
    m, k = cell % len(table), cell // len(table)
    u, base = table[m], []
    for a in range(D):
        base.append((k % nc[:, a].long()).double())
        k = k // nc[:, a].long()
    base = torch.stack(base, 1)
    if D == 3:
        odd = (base.sum(1) % 2) == 1
        u = torch.where(odd[:, None], torch.stack([1 - u[:, 1], u[:, 0], u[:, 2]], 1), u)
    return (base + u) / nc


def _series(A, x, terms=14):
    """v0, M v0 / 2, ...: the flow of x' = M x + b is x + sum_k s^(k+1) w_k."""
    M, b = A[..., :-1], A[..., -1]
    w = [(M * x[:, None, :]).sum(2) + b]
    for k in range(1, terms):
        w.append((M * w[-1][:, None, :]).sum(2) / (k + 1))
    return w


def _along(x, w, s):
    acc = w[-1]
    for k in range(len(w) - 2, -1, -1):
        acc = acc * s[:, None] + w[k]
    return x + acc * s[:, None]


@torch.no_grad()
def _pieces(x, nc, base, A, speed):
    """The pieces of each trajectory for time 1 that lie in one cell each: (points, row of A, duration) per step."""
    def stays(end, ns, cell, inner):
        # a hair outside is still inside: a point that goes along a face is not tossed from side to side by rounding
        return _cells(end + 1e-11 * (inner - end), ns) == cell

    x = x.clone()
    left = torch.ones(x.shape[0], dtype=F64, device=x.device)
    at = torch.arange(x.shape[0], device=x.device)
    got = []
    for _ in range(400):
        xs, ns, bs = x[at], nc[at], base[at]
        cell = _cells(xs, ns)
        row = bs + cell
        w = _series(A[row], xs)
        h = torch.minimum(left[at], speed[row])
        end = _along(xs, w, h)
        inner = _inner(cell, ns)
        out = (~stays(end, ns, cell, inner)).nonzero()[:, 0]
        if out.numel():  # the time at which it leaves, between one at which it is in and one at which it is out
            xo, no, co, ro, wo = xs[out], ns[out], cell[out], inner[out], [v[out] for v in w]
            lo, hi = torch.zeros_like(h[out]), h[out].clone()
            for _ in range(46):
                mid = 0.5 * (lo + hi)
                inside = stays(_along(xo, wo, mid), no, co, ro)
                lo, hi = torch.where(inside, mid, lo), torch.where(inside, hi, mid)
            h[out] = hi
            end = _along(xs, w, h)
        got.append((at, row, h))
        x[at] = end
        left[at] = left[at] - h
        at = at[left[at] > 1e-13]
        if not at.numel():
            return got
    return got


def _flow(x, nc, base, A, speed):
    """The points after time 1, differentiable in x and A: a field that is continuous across the cells' faces leaves no
    derivative of the crossing times."""
    for at, row, h in _pieces(x.detach(), nc, base, A.detach(), speed):
        xs = x[at]
        x = x.index_put((at,), _along(xs, _series(A[row], xs), h))
    return x


def _speed(A):
    """The longest piece of each row of A: its series converges fast, and no excursion is jumped over."""
    return (0.3 / A[..., :-1].reshape(A.shape[0], -1).norm(dim=1).clamp(min=1e-9)).clamp(max=0.125)


def _sample(data, off, stride, size, channels, x):
    """Linear interpolation [N, channels] of flat data at x [N, D]: sizes [N, D], one channel's values `stride` apart."""
    D = x.shape[1]
    p = x * (size - 1)
    lo = p.floor()
    i0 = torch.minimum(lo.clamp(min=0), size - 1)
    i1 = torch.minimum((lo + 1).clamp(min=0), size - 1)
    f = p - i0
    ch = torch.arange(channels, device=x.device)
    total = 0
    for corner in range(2 ** D):
        place, weight = torch.zeros_like(off), 1.0
        for a in range(D):
            up = (corner >> a) & 1
            place = place * size[:, a].long() + (i1 if up else i0)[:, a].long()
            weight = weight * (f[:, a] if up else 1 - f[:, a])
        total = total + weight[:, None] * data[off[:, None] + place[:, None] + ch * stride[:, None]]
    return total


def _mesh_point(t, out):
    """Coordinates [N, D] of output index t (last axis fastest) of grids `out` [N, D], with a float32 grid's values."""
    D, c = out.shape[1], []
    t = t.clone()
    for a in range(D - 1, -1, -1):
        c.append(t % out[:, a])
        t = t // out[:, a]
    i = torch.stack(c[::-1], 1)
    lines = {int(s): torch.linspace(0, 1, int(s), device=t.device).double() for s in out.unique().tolist()}
    x = torch.zeros(i.shape, dtype=F64, device=t.device)
    for s, line in lines.items():
        x = torch.where(out == s, line[i.clamp(max=s - 1)], x)
    return x


def _exact_data(nd, stages, data, off, size, channels, out, up, wants_data):
    """Flat problems of one dimension: out, dL/ddata (flat, as data) and dL/dA of each stage.  stages: [(A rows, first
    row of each problem, cells of each)]; off, size, out: per problem.  `up` None: no gradients."""
    dev = data.device
    npts = out.prod(1)
    first = torch.cumsum(npts, 0) - npts
    total = int(npts.sum())
    As = [A.clone().requires_grad_(up is not None) for A, _, _ in stages]
    speeds = [_speed(A.detach()) for A in As]
    data = data.clone().requires_grad_(up is not None and wants_data)
    result = torch.zeros(total * channels, dtype=F64, device=dev)
    for p0 in range(0, total, 1 << 20):
        t = torch.arange(p0, min(p0 + (1 << 20), total), device=dev)
        k = torch.searchsorted(first, t, right=True) - 1
        x = _mesh_point(t - first[k], out[k])
        with torch.set_grad_enabled(up is not None):
            for (_, row0, nc), A, sp in zip(stages, As, speeds):
                x = _flow(x, nc[k], row0[k], A, sp)
            v = _sample(data, off[k], size[k].prod(1), size[k].double(), channels, x)
            place = first[k][:, None] * channels + torch.arange(channels, device=dev) * npts[k][:, None] + (t - first[k])[:, None]
            result[place] = v.detach()
            if up is not None:
                (v * up[place]).sum().backward()
    return result, data.grad, [A.grad for A in As]


def _basis(T):
    p = T.get_params()
    return torch.as_tensor(p.basis).to("cuda", F64), p.ndim, p.nC


def exact(case, seed):
    s = prepare(case, seed)
    if s["kind"] == "ragged":
        return _exact_ragged(s)
    B, nd, nC = _basis(s["T"])
    n = case["n"]
    thetas = [t.detach().double() for t in s["thetas"]]
    A = [(t @ B.t()).reshape(n * nC, nd, nd + 1) for t in thetas]
    nc = torch.tensor(_ints(case["tess"]), dtype=F64, device="cuda")
    if s["kind"] == "numeric":
        return _exact_numeric(s, case, A[0].reshape(n, nC, nd, nd + 1), B, nc)
    row0 = torch.arange(n, device="cuda") * nC
    if s["kind"] in ("data", "chain"):
        data = s["data"].detach().double()
        C = data.shape[1]
        off = torch.arange(n, device="cuda") * (data.numel() // n)
        shape = torch.tensor(list(data.shape[2:]), device="cuda").expand(n, nd)
        out = torch.tensor(s["out"], device="cuda").expand(n, nd)
        up = s["upstream"].double().reshape(-1) if s["wrt"] else None
        res, gdata, gA = _exact_data(nd, [(a, row0, nc.expand(n, nd)) for a in A], data.reshape(-1), off, shape, C, out,
                                     up, s["data"].requires_grad)
        back = [res.reshape((n, C) + tuple(s["out"]))]
        if s["thetas"][0].requires_grad:
            back += [g.reshape(n, -1) @ B for g in gA]
        if s["data"].requires_grad:
            back.append(gdata.reshape(data.shape))
        return back
    grid = s["grid"].detach().double()
    P = grid.shape[-1]
    leaf = grid.clone().requires_grad_(bool(s["wrt"]))
    a = A[0].clone().requires_grad_(bool(s["wrt"]))
    with torch.set_grad_enabled(bool(s["wrt"])):
        x = (leaf if leaf.dim() == 3 else leaf.expand(n, nd, P)).permute(0, 2, 1).reshape(n * P, nd)
        y = _flow(x, nc.expand(n * P, nd), row0.repeat_interleave(P), a, _speed(a.detach()))
        y = y.reshape(n, P, nd).permute(0, 2, 1)
    back = [y.detach()]
    if s["wrt"]:
        (y * s["upstream"].double()).sum().backward()
        back += [a.grad.reshape(n, -1) @ B] if s["thetas"][0].requires_grad else []
        back += [leaf.grad] if s["grid"].requires_grad else []
    return back


def _exact_ragged(s):
    b, probs = s["batch"], s["probs"]
    flat = {k: torch.zeros(getattr(b, k).numel(), dtype=F64, device="cuda") for k in ("out", "grad_theta", "grad_data")}
    for nd in (1, 2):
        ids = [i for i, (T, _, _, _) in enumerate(probs) if T.get_params().ndim == nd]
        if not ids:
            continue
        mats = [_basis(probs[i][0])[0] for i in ids]
        rows = [(B @ b.theta_views[i].double()).reshape(-1, nd, nd + 1) for i, B in zip(ids, mats)]
        count = torch.tensor([r.shape[0] for r in rows], device="cuda")
        nc = torch.tensor([probs[i][0].get_params().nc for i in ids], dtype=F64, device="cuda")
        size = torch.tensor([probs[i][2] for i in ids], device="cuda")
        C = probs[ids[0]][1]
        data = torch.cat([b.data_views[i].reshape(-1) for i in ids]).double()
        up = torch.cat([b.grad_out_views[i].reshape(-1) for i in ids]).double()
        per = size.prod(1) * C
        off = torch.cumsum(per, 0) - per
        res, gdata, gA = _exact_data(nd, [(torch.cat(rows), torch.cumsum(count, 0) - count, nc)], data, off, size, C, size,
                                     up, True)
        r0 = 0
        for i, B, r, o, m in zip(ids, mats, rows, off.tolist(), per.tolist()):
            for key, view, value in (("out", b.out_views[i], res[o:o + m]), ("grad_data", b.grad_data_views[i], gdata[o:o + m]),
                                     ("grad_theta", b.grad_theta_views[i], gA[0][r0:r0 + r.shape[0]].reshape(-1) @ B)):
                at = view.storage_offset()
                flat[key][at:at + value.numel()] = value
            r0 += r.shape[0]
    return flat


def _exact_numeric(s, case, A, B, nc):
    """The fixed-step scheme: expm(A / steps) per cell and step, and midpoint steps of the point and its derivatives."""
    n, nC, nd, _ = A.shape
    steps, P = case["steps"], s["grid"].shape[-1]
    hom = torch.zeros(n, nC, nd + 1, nd + 1, dtype=F64, device="cuda")
    hom[:, :, :nd] = A
    trel = torch.matrix_exp(hom / steps)[:, :, :nd].reshape(n * nC, nd, nd + 1)
    x0 = s["grid"].double().t().repeat(n, 1)  # [n * P, nd]
    base = (torch.arange(n, device="cuda") * nC).repeat_interleave(P)
    ncs = nc.expand(n * P, nd)

    def apply(M, p):
        return (M[..., :-1] * p[..., None, :]).sum(-1) + M[..., -1]

    x = x0
    for _ in range(steps):
        x = apply(trel[base + _cells(x, ncs)], x)
    back = [x.reshape(n, P, nd).permute(0, 2, 1)]
    if not s["wrt"]:
        return back
    Bk = B.t().reshape(-1, nC, nd, nd + 1)
    rows, h = A.reshape(n * nC, nd, nd + 1), 1.0 / steps
    g = s["upstream"].double().permute(0, 2, 1).reshape(n * P, nd)
    p = x0
    q = torch.zeros(Bk.shape[0], n * P, nd, dtype=F64, device="cuda")
    for _ in range(steps):
        cell = _cells(p, ncs)
        M, N = rows[base + cell], Bk[:, cell]
        pm = p + 0.5 * h * apply(M, p)
        lin = M[:, :, :-1]
        qm = q + 0.5 * h * (apply(N, p) + (lin * q[..., None, :]).sum(-1))
        q = q + h * (apply(N, pm) + (lin * qm[..., None, :]).sum(-1))
        p = p + h * apply(M, pm)
    grad = (q * g).reshape(-1, n, P, nd).sum((2, 3)).t()
    return back + [grad]
