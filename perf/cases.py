"""The work that programs built on this framework spend their time in, as cases to be timed.

A case is one call (or one job) at one size: projectors of tilt scans and of general polar
grids in both directions, the normal operator of the solvers, a preconditioned CG solve and
a whole reconstruction job.  Sizes run from the smallest volumes of the test configurations
to the precision-study benchmark; odd and even lengths, one to three datasets, several
kernel widths.  Inputs are made from a seed; `exact` restates each call in 64 bits with
plain torch.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import lamino_amd as la
from lamino_amd import _lib

DEV = "cuda"
TWO_PI = 2.0 * math.pi


# ------------------------------------------------------------------------------ the cases


def _case(op, n, det, proj, sets=1, tilt=30.0, eps=1e-5, iters=0, name=None):
    c = {"op": op, "n1": n[0], "n2": n[1], "n3": n[2], "rows": det[0], "cols": det[1], "proj": proj, "sets": sets,
         "tilt": tilt, "eps": eps, "iters": iters}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the projectors of the plain-CG configuration: a few hundred microseconds, launch-bound
        _case("forward", (89, 21, 89), (89, 89), 90, name="forward_small"),
        _case("adjoint", (89, 21, 89), (89, 89), 90, name="adjoint_small"),
        # an even-sized volume and detector (no odd-ification), a tighter tolerance (wider kernel)
        _case("forward", (100, 24, 96), (120, 128), 75, tilt=40.0, eps=1e-6, name="forward_even"),
        _case("adjoint", (100, 24, 96), (120, 128), 75, tilt=40.0, eps=1e-6, name="adjoint_even"),
        # the split-Bregman configuration: two datasets of 180 projections, data simulation
        # and the backprojection that every job starts with
        _case("forward", (179, 43, 179), (305, 305), 180, sets=2, tilt=35.0, name="forward_medium"),
        _case("adjoint", (179, 43, 179), (305, 305), 180, sets=2, tilt=35.0, name="adjoint_medium"),
        # the precision-study configuration, the headline benchmark's step
        _case("forward", (359, 71, 359), (615, 615), 360, sets=3, name="forward_large"),
        _case("adjoint", (359, 71, 359), (615, 615), 360, sets=3, name="adjoint_large"),
        # the reference's own PolarGrid(angles, rows, cols, gamma): the tilt varies with the angle
        _case("polar", (127, 31, 127), (181, 181), 120, name="polar_roundtrip"),
        # one application of the solvers' normal operator at the precision-study size
        _case("normal", (359, 71, 359), (615, 615), 360, sets=3, name="normal_large"),
        # preconditioned CG on the normal operator at the split-Bregman size
        _case("cg", (179, 43, 179), (305, 305), 180, sets=2, tilt=35.0, iters=10, name="cg_medium"),
        # a whole qGGMRF reconstruction, host projections to host volume
        _case("job3", (63, 15, 63), (63, 63), 90, sets=2, iters=10, name="job_qggmrf"),
    ]


def draw(rng):
    def logu(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["forward", "adjoint", "forward", "adjoint", "polar", "normal", "cg", "job1", "job2", "job3"])
    big = {"forward": 359, "adjoint": 359, "polar": 180, "normal": 359, "cg": 240, "job1": 127, "job2": 100,
           "job3": 90}[op]
    n3 = logu(40, big)
    n1 = max(20, min(big, n3 + rng.randint(-9, 9)))
    n2 = max(7, int(n3 * rng.uniform(0.15, 0.28)))
    f = rng.uniform(1.0, 1.71)
    cols = int(n3 * f)
    rows = max(30, min(615, cols + rng.randint(-5, 5)))
    if op.startswith("job"):   # jobs pad by themselves and take odd sizes
        n1, n2, n3 = n3 | 1, n2 | 1, n3 | 1
        rows = cols = n3
    proj = logu(30, 180 if op in ("polar", "job1", "job2", "job3") else 360)
    sets = 1 if op == "polar" else rng.randint(1, 3)
    eps = rng.choice([1e-5, 1e-5, 1e-5, 1e-4, 1e-6]) if op in ("forward", "adjoint", "polar") else 1e-5
    iters = rng.randint(3, 12) if op in ("cg", "job1", "job2", "job3") else 0
    return _case(op, (n1, n2, n3), (rows, cols), proj, sets, round(rng.uniform(25.0, 40.0), 2), eps, iters)


# ------------------------------------------------------------------------------ inputs


def _gen(seed, stream):
    g = torch.Generator(device="cpu")
    g.manual_seed((int(seed) * 1000003 + stream * 7919 + 17) % (1 << 62))
    return g


def _angles(case, seed):
    """[(alpha, gamma)] per dataset (numpy float64): a tilt scan each, datasets 45 degrees apart,
    or for a general polar grid the reference's angles at one gamma."""
    P = case["proj"]
    off = float(torch.rand(1, generator=_gen(seed, 1), dtype=torch.float64)) * 0.1
    j = np.arange(P, dtype=np.float64)
    if case["op"] == "polar":
        return [(np.pi * (j + off) / P, np.full(P, math.radians(30.0) + off))]
    return [(np.full(P, math.radians(case["tilt"])), TWO_PI * j / P + math.radians(45.0 * s) + off)
            for s in range(case["sets"])]


def _smooth(shape, seed, stream, blobs=24):
    """Sum of separable Gaussian blobs on the last axes of `shape` plus 1 % noise, float32 on the GPU."""
    g = _gen(seed, stream)
    axes = shape[1:]
    out = torch.zeros(shape, dtype=torch.float32, device=DEV)
    amp = (torch.rand(blobs, shape[0], generator=g) * 2 - 1).to(DEV)
    prof = []
    for n in axes:
        c = (0.2 + 0.6 * torch.rand(blobs, generator=g)) * n
        w = (0.02 + 0.08 * torch.rand(blobs, generator=g)) * n + 0.8
        t = torch.arange(n, dtype=torch.float32)
        prof.append(torch.exp(-0.5 * ((t[None] - c[:, None]) / w[:, None]) ** 2).to(DEV))
    if len(axes) == 3:
        zy = prof[0][:, :, None] * prof[1][:, None, :]
        for i in range(shape[0]):
            out[i] = torch.matmul((zy * amp[:, i, None, None]).reshape(blobs, -1).t(), prof[2]).reshape(axes)
    else:
        out = torch.matmul((amp.t()[:, :, None] * prof[0][None]).transpose(1, 2).contiguous(), prof[1])
    gd = torch.Generator(device=DEV)
    gd.manual_seed((int(seed) * 1000003 + stream) % (1 << 62))
    out += 0.01 * torch.randn(shape, generator=gd, device=DEV)
    return out.contiguous()


def _inset(x):
    """Zero outside the centred part that the reference's padding leaves (PAD_FACTOR 1.4142)."""
    for d in range(1, x.dim()):
        n = x.shape[d]
        e = (n - int(n / 1.4142)) // 2
        if e > 0:
            x.narrow(d, 0, e).zero_()
            x.narrow(d, n - e, e).zero_()
    return x


def _volume(case, seed):
    return _inset(_smooth((3, case["n1"], case["n2"], case["n3"]), seed, 2))


def _projections(case, seed, k):
    p = _smooth((case["proj"], case["rows"], case["cols"]), seed, 10 + k)
    return _inset(p / p.max())


# ------------------------------------------------------------------------------ the calls


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _comps(v):
    return [_ptr(v[i]) for i in range(3)]


def _dims(case):
    return (ctypes.c_int64 * 3)(case["n1"], case["n2"], case["n3"])


def _vec(v):
    return (ctypes.c_void_p * 3)(*[v[i].data_ptr() for i in range(3)])


def _grids(case, seed):
    R, C = case["rows"], case["cols"]
    if case["op"] == "polar":
        al, ga = _angles(case, seed)[0]
        return [la.PolarGrid(al, R, C, float(ga[0]))]
    return [la.PolarGrid.per_projection(al, ga, R, C) for al, ga in _angles(case, seed)]


def prepare(case, seed):
    op = case["op"]
    s = {"case": case, "ctx": la.default_context(), "dims": _dims(case)}
    vol = (3, case["n1"], case["n2"], case["n3"])
    stack = (case["proj"], case["rows"], case["cols"])
    if op.startswith("job"):
        ang = _angles(case, seed)
        s["datasets"] = [(_projections(case, seed, k).abs().cpu().numpy(), a, g) for k, (a, g) in enumerate(ang)]
        s["params"] = la.ReconParams(max_iters=case["iters"], inner_iters=3, mu=0.0 if op == "job3" else 10.0,
                                     tol=0.0, xtol=0.0, eps=case["eps"])
        return s
    grids = _grids(case, seed)
    s["grids"] = grids
    if op in ("normal", "cg"):
        s["op"] = la.ToeplitzOperator(grids, vol[1:])
        s["x"] = _volume(case, seed)
        s["out"] = torch.empty(vol, device=DEV)
        s["zero"] = torch.zeros(vol, device=DEV)
        s["A"] = _lib.OP_FN(ctypes.cast(s["ctx"].lib.lam_toep_op, ctypes.c_void_p).value)
        return s
    s["handles"] = (ctypes.c_void_p * len(grids))(*[g.h for g in grids])
    if op in ("forward", "polar"):
        s["m"] = _volume(case, seed)
        s["proj"] = [torch.empty(stack, device=DEV) for _ in grids]
    else:
        s["proj"] = [_projections(case, seed, k) for k in range(len(grids))]
    if op in ("adjoint", "polar"):
        s["vol"] = torch.empty(vol, device=DEV)
    s["stacks"] = (ctypes.c_void_p * len(grids))(*[p.data_ptr() for p in s["proj"]])
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    op, lib = case["op"], ctx.lib
    if op.startswith("job"):
        job = {"job1": la.MBIR1, "job2": la.MBIR2, "job3": la.MBIR3}[op]
        return job(s["datasets"], (case["n1"], case["n2"], case["n3"]), s["params"])
    dims, eps = s["dims"], case["eps"]
    if op == "normal":
        _lib.check(lib.lam_toep_apply(s["op"].h, _vec(s["x"]), _vec(s["out"]), 0.0))
        return s["out"]
    if op == "cg":
        it = ctypes.c_int64()
        _lib.check(lib.lam_cgsolver(ctx.h, dims, s["A"], s["op"].h, _vec(s["x"]), _vec(s["zero"]), case["iters"], 0.0,
                                    _vec(s["out"]), ctypes.byref(it)))
        return s["out"]
    if op == "polar":   # data simulation on the grid, then its backprojection
        g = s["grids"][0]
        _lib.check(lib.lam_forward(ctx.h, g.h, dims, eps, *_comps(s["m"]), _ptr(s["proj"][0])))
        _lib.check(lib.lam_adjoint(ctx.h, g.h, dims, eps, _ptr(s["proj"][0]), *_comps(s["vol"])))
        return [s["proj"][0], s["vol"]]
    if op == "forward":
        _lib.check(lib.lam_forward_multi(ctx.h, s["handles"], len(s["grids"]), dims, eps, *_comps(s["m"]),
                                         s["stacks"]))
        return s["proj"]
    _lib.check(lib.lam_adjoint_multi(ctx.h, s["handles"], len(s["grids"]), dims, eps, s["stacks"], *_comps(s["vol"]),
                                     0))
    return s["vol"]


def work(case):
    nv = case["n1"] * case["n2"] * case["n3"]
    M = case["proj"] * case["rows"] * case["cols"] * case["sets"]
    w = 4 if case["eps"] >= 1e-3 else 6 if case["eps"] >= 9e-6 else 8
    nf, lg = 8 * nv, 8 * nv
    fft = lambda n: 5.0 * n * math.log2(n)  # noqa: E731
    # one pass of a projector: the transform of the three components on the fine grid and the
    # kernel's taps at half of the (Hermitian) points, and the planes' own transforms
    taps = w * w * (w if case["op"] == "polar" else 1)
    projector = 3 * fft(nf) + M / 2 * taps * 12 + M / 2 * 5 * math.log2(max(2, case["rows"] * case["cols"]))
    normal = 2 * 3 * fft(lg) / 2 + lg / 2 * 30
    if case["op"] == "normal":
        return {"bytes": 24 * nv + 24 * (lg // 2), "flops": normal}
    if case["op"] == "cg":
        return {"bytes": case["iters"] * (24 * nv + 24 * (lg // 2)), "flops": case["iters"] * (normal + 6 * fft(nv))}
    if case["op"].startswith("job"):
        inner = {"job1": 1, "job2": 3, "job3": 2}[case["op"]] * case["iters"]
        return {"bytes": 4 * M + 12 * nv, "flops": 3 * M * w * w * 6 + inner * 3 * (normal + 6 * fft(nv))}
    k = 2 if case["op"] == "polar" else 1
    return {"bytes": k * (12 * nv + 4 * M), "flops": k * projector}


# ------------------------------------------------------------------------------ 64-bit restatement


def _phase(a, b):
    """exp(i a b) of two float64 vectors, as an outer product (complex128)."""
    t = a[:, None] * b[None, :]
    return torch.complex(torch.cos(t), torch.sin(t))


def _modes(n):
    return torch.arange(n, dtype=torch.float64, device=DEV) - n // 2


class _Plane:
    """One projection's phases over the upper half of its rows (the rest follow by symmetry)."""

    def __init__(self, case, a, g):
        R, C = case["rows"], case["cols"]
        self.J = (R + 1) // 2
        qx = (torch.arange(C, dtype=torch.float64, device=DEV) - (C - 1) / 2) * (TWO_PI / C)
        qy = (torch.arange(self.J, dtype=torch.float64, device=DEV) - (R - 1) / 2) * (TWO_PI / R)
        z, y, x = _modes(case["n1"]), _modes(case["n2"]), _modes(case["n3"])
        self.xk, self.zk = _phase(x, qx * math.cos(g)), _phase(z, qx * -math.sin(g))
        self.xj, self.zj = _phase(x, qy * math.cos(a) * math.sin(g)), _phase(z, qy * math.cos(a) * math.cos(g))
        self.yj = _phase(y, qy * -math.sin(a))
        self.d = (math.sin(g) * math.sin(a), math.cos(a), math.cos(g) * math.sin(a))


def _rows(case):
    return max(1, (1 << 25) // (case["n1"] * max(case["n3"], case["cols"])))


def _shift(x, inverse):
    r, c = x.shape[-2:]
    up = (-(-r // 2), -(-c // 2)) if inverse else (r // 2, c // 2)
    return torch.roll(x, (-up[0], -up[1]), dims=(-2, -1))


def _forward64(case, m, alpha, gamma):
    n1, n2, n3, R, C = (case[k] for k in ("n1", "n2", "n3", "rows", "cols"))
    m = m.double()
    out = torch.empty((len(alpha), R, C), dtype=torch.float64, device=DEV)
    shared = bool((alpha == alpha[0]).all())
    part = None
    for p, (a, g) in enumerate(zip(alpha, gamma)):
        pl = _Plane(case, float(a), float(g))
        if part is None or not shared:
            vols = [m[i].transpose(0, 1).reshape(n2, n1 * n3).to(torch.complex128) for i in range(3)]
            if shared:
                part = [torch.matmul(pl.yj.conj().t(), v).reshape(pl.J, n1, n3) for v in vols]
            else:
                v = sum(d * u for d, u in zip(pl.d, vols))
                part = [torch.matmul(pl.yj.conj().t(), v).reshape(pl.J, n1, n3)]
        c = torch.empty((R, C), dtype=torch.complex128, device=DEV)
        for j in range(0, pl.J, _rows(case)):
            s = slice(j, min(pl.J, j + _rows(case)))
            b = sum(d * u[s] for d, u in zip(pl.d, part)) if shared else part[0][s]
            b = b * pl.zj.conj().t()[s, :, None] * pl.xj.conj().t()[s, None, :]
            t = torch.matmul(b.reshape(-1, n3), pl.xk.conj().resolve_conj()).reshape(-1, n1, C)
            c[s] = (t * pl.zk.conj()[None]).sum(1)
        c[R - pl.J:] = torch.where(torch.arange(R - pl.J, R, device=DEV)[:, None] >= pl.J,
                                   c[:pl.J].flip(0, 1).conj(), c[R - pl.J:])
        out[p] = _shift(torch.fft.ifft2(_shift(c, False)), True).real
    return out


def _adjoint64(case, proj, alpha, gamma, acc):
    n1, n2, n3, R, C = (case[k] for k in ("n1", "n2", "n3", "rows", "cols"))
    shared = bool((alpha == alpha[0]).all())
    part, pl = None, None
    for p, (a, g) in enumerate(zip(alpha, gamma)):
        pl = _Plane(case, float(a), float(g))
        c = _shift(torch.fft.fft2(_shift(proj[p].to(torch.complex128), False)), True)
        v = (c + c.flip(0, 1).conj())[:pl.J]
        if R % 2:
            v[-1] *= 0.5     # the middle row holds both points of each pair
        h = [torch.zeros((pl.J, n1, n3), dtype=torch.complex128, device=DEV) for _ in range(3 if part is None else 0)]
        part = part or h
        for j in range(0, pl.J, _rows(case)):
            s = slice(j, min(pl.J, j + _rows(case)))
            t = (v[s][:, None, :] * pl.zk[None]).reshape(-1, C)
            b = torch.matmul(t, pl.xk.t().contiguous()).reshape(-1, n1, n3)
            b = b * pl.zj.t()[s, :, None] * pl.xj.t()[s, None, :]
            for i in range(3):
                part[i][s] += pl.d[i] * b
        if not shared:
            _rows_to_volume(part, pl, acc, n1, n2, n3, R * C)
            part = None
    if shared:
        _rows_to_volume(part, pl, acc, n1, n2, n3, R * C)


def _rows_to_volume(part, pl, acc, n1, n2, n3, scale):
    for i in range(3):
        f = torch.matmul(pl.yj, part[i].reshape(pl.J, n1 * n3)).real.reshape(n2, n1, n3)
        acc[i] += f.transpose(0, 1) / scale


def _dirichlet(v, n):
    """sin(pi v) / sin(pi v / n), with its limit where the denominator vanishes."""
    den = torch.sin(math.pi * torch.remainder(v / n, 2.0))
    num = torch.sin(math.pi * torch.remainder(v, 2.0))
    m = torch.round(v / n)
    lim = torch.where(torch.remainder(m * (n - 1), 2.0) == 0, float(n), -float(n)).to(v.dtype)
    return torch.where(den.abs() < 1e-10, lim, num / torch.where(den.abs() < 1e-10, torch.ones_like(den), den))


class _Normal64:
    """sum_g adjoint_g(forward_g(x)) as a convolution with its closed-form kernel."""

    PAIRS = ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))

    def __init__(self, case, seed):
        n = (case["n1"], case["n2"], case["n3"])
        R, C = case["rows"], case["cols"]
        self.n = n
        self.L = tuple(self._length(2 * v - 1) for v in n)
        dz, dy = (torch.arange(-(v - 1), v, dtype=torch.float64, device=DEV) for v in n[:2])
        dx = torch.arange(0, n[2], dtype=torch.float64, device=DEV)
        ker = [torch.zeros((2 * n[0] - 1, 2 * n[1] - 1, n[2]), dtype=torch.float64, device=DEV) for _ in self.PAIRS]
        for alpha, gamma in _angles(case, seed):
            for a, g in zip(alpha, gamma):
                d = (math.sin(g) * math.sin(a), math.cos(a), math.cos(g) * math.sin(a))
                u = dx[None, :] * math.cos(g) - dz[:, None] * math.sin(g)
                v = dx[None, :] * (math.cos(a) * math.sin(g)) + dz[:, None] * (math.cos(a) * math.cos(g))
                t = _dirichlet(v[:, None, :] - dy[None, :, None] * math.sin(a), R)
                t *= (_dirichlet(u, C) / (R * C))[:, None, :]
                for q, (i, k) in enumerate(self.PAIRS):
                    ker[q].add_(t, alpha=d[i] * d[k])
        self.hat = []
        for q in range(6):
            full = torch.zeros(self.L, dtype=torch.float64, device=DEV)
            iz, iy = torch.remainder(dz.long(), self.L[0]), torch.remainder(dy.long(), self.L[1])
            ix = dx.long()
            full[iz[:, None, None], iy[None, :, None], ix[None, None, :]] = ker[q]
            full[torch.remainder(-iz, self.L[0])[:, None, None], torch.remainder(-iy, self.L[1])[None, :, None],
                 torch.remainder(-ix, self.L[2])[None, None, :]] = ker[q]
            ker[q] = None
            self.hat.append(torch.fft.rfftn(full).real)

    @staticmethod
    def _length(n):
        while True:
            r = n
            for p in (2, 3, 5):
                while r % p == 0:
                    r //= p
            if r == 1:
                return n
            n += 1

    def __call__(self, x):
        X = [torch.fft.rfftn(x[i], s=self.L) for i in range(3)]
        out = torch.empty_like(x)
        for i in range(3):
            Y = sum(self.hat[self.PAIRS.index((min(i, k), max(i, k)))] * X[k] for k in range(3))
            out[i] = torch.fft.irfftn(Y, s=self.L)[:self.n[0], :self.n[1], :self.n[2]]
        return out


def _ramp64(x):
    fy = torch.fft.fftfreq(x.shape[-2], dtype=torch.float64, device=DEV)
    fx = torch.fft.rfftfreq(x.shape[-1], dtype=torch.float64, device=DEV)
    f = torch.sqrt(fy[:, None] ** 2 + fx[None, :] ** 2)
    return torch.fft.irfft2(torch.fft.rfft2(x) * f, s=x.shape[-2:])


def _cg64(A, b, iters):
    x = torch.zeros_like(b)
    r = b.clone()
    z = _ramp64(r)
    p = z.clone()
    rs = (z * r).sum()
    for _ in range(iters):
        Ap = A(p)
        alpha = rs / (p * Ap).sum()
        x += alpha * p
        r -= alpha * Ap
        z = _ramp64(r)
        new = (z * r).sum()
        p = z + (new / rs) * p
        rs = new
    return x


def exact(case, seed):
    op = case["op"]
    if op.startswith("job"):
        return None   # tens of solver iterations on an iterated operator
    ang = _angles(case, seed)
    if op == "normal":
        return _Normal64(case, seed)(_volume(case, seed).double())
    if op == "cg":
        return _cg64(_Normal64(case, seed), _volume(case, seed).double(), case["iters"])
    vol = (3, case["n1"], case["n2"], case["n3"])
    if op == "forward":
        m = _volume(case, seed)
        return [_forward64(case, m, a, g) for a, g in ang]
    acc = torch.zeros(vol, dtype=torch.float64, device=DEV)
    if op == "polar":
        m = _volume(case, seed)
        p = _forward64(case, m, *ang[0])
        _adjoint64(case, p, *ang[0], acc)
        return [p, acc]
    for k, (a, g) in enumerate(ang):
        _adjoint64(case, _projections(case, seed, k).double(), a, g, acc)
    return acc
