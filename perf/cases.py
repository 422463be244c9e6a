"""The solves and time steps this library's speed is measured on.

Every case goes through the public Python entry points (fdm_amd, fdm_amd.serve),
on the domain [-pi, pi] per axis with the reference's spacing and length
convention (h = 2 pi / n, l = 2 pi + h on a Dirichlet axis, l = 2 pi on a
periodic one).  Right-hand sides are the discrete Laplacian of a field drawn
uniform in [-1, 1] with zero boundary, which is what the library's benchmark,
its batched and served workloads and its tests solve; the periodic solve takes
a particle-mesh density (a field with a mean), as the reference's n-body code
hands it one.

A case is a dict of plain values.  `kind` says which entry point it drives:
  cube    LaplCube.solve (batch 1) or solve_batch, device arrays
  pcube   the same, periodic on every axis
  rect    LaplRect.solve / solve_batch, device arrays
  host    LaplCube.solve on host arrays, the drop-in class's own call
  group   serve.Group: many problems of uneven shapes in one recorded sequence
  serve   serve.Server: a burst of requests submitted and waited for
  ns      NSCube.step: steps of the lid-driven cavity
"""
import ctypes
import math
import random

import numpy as np
import torch

import fdm_amd
from fdm_amd import hip, serve

PI2 = 2.0 * math.pi


def listed():
    return [
        # one solve of the smallest cube in use (32 per axis on the reference's
        # count): three short launches, latency only
        {"name": "cube31_f64", "kind": "cube", "prec": "f64", "nx": 31, "ny": 31, "nz": 31, "batch": 1},
        # one LaplCube<float> solve at the size most code runs (half a plane per CU)
        {"name": "cube127_f32", "kind": "cube", "prec": "f32", "nx": 127, "ny": 127, "nz": 127, "batch": 1},
        # the headline batch, in plain double and in FP32 with FP64 refinement to 1e-10
        {"name": "cube127_f64_b32", "kind": "cube", "prec": "f64", "nx": 127, "ny": 127, "nz": 127, "batch": 32},
        {"name": "cube127_refine_b32", "kind": "cube", "prec": "refine", "nx": 127, "ny": 127, "nz": 127,
         "batch": 32},
        # the single large solve, both precisions
        {"name": "cube255_f64", "kind": "cube", "prec": "f64", "nx": 255, "ny": 255, "nz": 255, "batch": 1},
        {"name": "cube255_refine", "kind": "cube", "prec": "refine", "nx": 255, "ny": 255, "nz": 255, "batch": 1},
        # the Poisson stage of a particle-mesh step (periodic, double)
        {"name": "periodic128_f64", "kind": "pcube", "prec": "f64", "nx": 128, "ny": 128, "nz": 128, "batch": 1},
        # the 2-D solver at the size its unit tests use
        {"name": "rect511_f64", "kind": "rect", "prec": "f64", "nx": 511, "ny": 511, "batch": 1},
        # 512 problems, each axis from {31, 63, 127}, a quarter of them 2-D
        {"name": "uneven512_refine", "kind": "group", "prec": "refine", "count": 512},
        # a burst of requests of that mix with some 255^3 among them
        {"name": "serve64_refine", "kind": "serve", "prec": "refine", "count": 64},
        # ten steps of the 127^3 cavity, refined pressure solve
        {"name": "cavity127_refine", "kind": "ns", "prec": "refine", "nx": 127, "ny": 127, "nz": 127, "steps": 10},
        # the drop-in's own call: host arrays in and out
        {"name": "host127_f64", "kind": "host", "prec": "f64", "nx": 127, "ny": 127, "nz": 127, "batch": 1},
    ]


MOST_POINTS = 32 * 127 ** 3   # of a drawn batch: the listed one's


def draw(rng: random.Random):
    kind = rng.choice(["cube", "cube", "cube", "pcube", "rect", "group", "serve", "ns", "host"])
    if kind in ("cube", "pcube", "host"):
        e = 0 if kind == "pcube" else 1
        prec = rng.choice(["f32", "f64"] if kind == "pcube" else ["f32", "f64", "refine"])
        if rng.random() < 0.5:
            n = [(1 << rng.randint(4, 8)) - e] * 3
        else:
            n = [(1 << rng.randint(4, 8)) - e for _ in range(3)]
        most = max(1, min(512, MOST_POINTS // (n[0] * n[1] * n[2])))
        batch = 1 if kind == "host" or rng.random() < 0.3 else int(round(math.exp(rng.uniform(0, math.log(most)))))
        return {"kind": kind, "prec": prec, "nx": n[0], "ny": n[1], "nz": n[2], "batch": max(1, batch)}
    if kind == "rect":   # LaplRect takes any number of points along x
        return {"kind": "rect", "prec": rng.choice(["f32", "f64", "refine"]),
                "nx": int(round(math.exp(rng.uniform(math.log(16), math.log(1024))))),
                "ny": (1 << rng.randint(4, 9)) - 1, "batch": int(round(math.exp(rng.uniform(0, math.log(64)))))}
    if kind == "group":
        return {"kind": "group", "prec": rng.choice(["f32", "f64", "refine"]),
                "count": int(round(math.exp(rng.uniform(math.log(16), math.log(320)))))}
    if kind == "serve":
        return {"kind": "serve", "prec": rng.choice(["f64", "refine"]),
                "count": int(round(math.exp(rng.uniform(math.log(4), math.log(64)))))}
    n = [(1 << rng.randint(4, 7)) - 1 for _ in range(3)]
    n.sort(reverse=True)   # the cavity needs nz <= nx
    return {"kind": "ns", "prec": rng.choice(["f64", "refine"]), "nx": n[0], "ny": n[1], "nz": n[2],
            "steps": rng.randint(1, 10)}


# ---- shapes and inputs ------------------------------------------------------
def _shapes(case):
    """Per problem (nx, ny, nz), nz = 0 for a rect; the same for every seed."""
    if case["kind"] in ("cube", "pcube", "host"):
        return [(case["nx"], case["ny"], case["nz"])] * case["batch"]
    if case["kind"] == "rect":
        return [(case["nx"], case["ny"], 0)] * case["batch"]
    rng = random.Random(3)
    out = []
    for i in range(case["count"]):
        if case["kind"] == "serve" and i % 20 == 7:   # 5% large
            out.append((255, 255, 255))
            continue
        s = tuple(rng.choice((31, 63, 127)) for _ in range(3))
        out.append(s[:2] + (0,) if rng.random() < 0.25 else s)
    return out


def _points(s):
    return s[0] * s[1] * max(1, s[2])


def _spacing(n, periodic):
    h = PI2 / n
    return h, (PI2 if periodic else PI2 + h)


def _stencil_steps(s, periodic):
    """1/h^2 per axis (x, y, z) of the operator the solver inverts: LaplCube uses
    the y spacing on an axis with as many points as y, which is the same here."""
    return [1.0 / _spacing(n, periodic)[0] ** 2 for n in s if n]


def _problem_rhs(s, dtype, g):
    """The discrete Laplacian of a uniform field on one shape, on the GPU."""
    dims = [n for n in reversed(s) if n]
    pad = torch.zeros([n + 2 for n in dims], dtype=torch.float64, device="cuda")
    core = tuple(slice(1, -1) for _ in dims)
    pad[core] = torch.rand(dims, dtype=torch.float64, device="cuda", generator=g) * 2 - 1
    f = torch.zeros(dims, dtype=torch.float64, device="cuda")
    for a, c in enumerate(reversed(_stencil_steps(s, False))):
        lo = tuple(slice(0, -2) if b == a else slice(1, -1) for b in range(len(dims)))
        hi = tuple(slice(2, None) if b == a else slice(1, -1) for b in range(len(dims)))
        f += (pad[lo] - 2 * pad[core] + pad[hi]) * c
    return f.to(dtype)


def _dtype(case):
    return torch.float32 if case["prec"] == "f32" else torch.float64


def _inputs(case, seed):
    """All right-hand sides of a case, back to back in one device tensor."""
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * seed + 17)
    shapes, dtype = _shapes(case), _dtype(case)
    flat = torch.empty(sum(_points(s) for s in shapes), dtype=dtype, device="cuda")
    at = 0
    for s in shapes:
        m = _points(s)
        if case["kind"] == "pcube":   # a density: positive, with a mean
            r = torch.rand(m, dtype=torch.float64, device="cuda", generator=g)
            flat[at:at + m] = (4.0 * math.pi * r * r).to(dtype)
        else:
            flat[at:at + m] = _problem_rhs(s, dtype, g).reshape(-1)
        at += m
    return flat


def _views(flat, shapes):
    at, out = 0, []
    for s in shapes:
        out.append(flat[at:at + _points(s)])
        at += _points(s)
    return out


def _plan(case):
    nx, ny = case["nx"], case["ny"]
    per = case["kind"] == "pcube"
    (dx, lx), (dy, ly) = _spacing(nx, per), _spacing(ny, per)
    if case["kind"] == "rect":
        return fdm_amd.LaplRect(dx, dy, lx, ly, nx, ny, precision=case["prec"])
    dz, lz = _spacing(case["nz"], per)
    return fdm_amd.LaplCube(dx, dy, dz, lx, ly, lz, nx, ny, case["nz"], precision=case["prec"], periodic=per)


def _problem(s, prec, ans, rhs):
    p = fdm_amd._prec(prec)
    (dx, lx), (dy, ly) = _spacing(s[0], False), _spacing(s[1], False)
    if not s[2]:
        return serve.rect_problem(dx, dy, lx, ly, s[0], s[1], ans.data_ptr(), rhs.data_ptr(), precision=p)
    dz, lz = _spacing(s[2], False)
    return serve.cube_problem(dx, dy, dz, lx, ly, lz, s[0], s[1], s[2], ans.data_ptr(), rhs.data_ptr(), precision=p)


# ---- the cavity's fields ----------------------------------------------------
NS_RE, NS_DT, NS_U0 = 250.0, 0.01, 1.0


def _ns_fields(case, seed):
    """A developed flow to continue from: the sum of a few smooth modes per
    velocity component plus small noise, and a pressure of its scale."""
    rng = np.random.default_rng(seed)
    shapes = fdm_amd.ns_shapes(case["nx"], case["ny"], case["nz"])
    out = {}
    for name, amp in (("u", 0.3), ("v", 0.3), ("w", 0.3), ("p", 0.05)):
        shape = shapes[name]
        a = 0.02 * amp * rng.uniform(-1, 1, shape)
        for _ in range(3):
            w = [np.sin(rng.integers(1, 5) * math.pi * np.linspace(0, 1, m) + 0.3 * rng.uniform()) for m in shape]
            a += amp * rng.uniform(-1, 1) * w[0][:, None, None] * w[1][None, :, None] * w[2][None, None, :]
        out[name] = a
    return out


class _DeviceField:
    """A device array of the library as torch sees it; holds its owner, whose
    end frees the memory."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8", "data": (ptr, False), "version": 3,
                                         "strides": None}


class _Fields(dict):
    """Views of a time-stepper's arrays, which live as long as the views' dict."""

    def __init__(self, ns, names):
        super().__init__((f, _ns_view(ns, f)) for f in names)
        self.ns = ns


def _ns_view(ns, name):
    ptr, count = ctypes.c_void_p(), ctypes.c_ulonglong()
    rc = fdm_amd.lib().fdmgpu_ns_info(ns._h, fdm_amd.NS_FIELDS.index(name), ctypes.byref(count), ctypes.byref(ptr))
    if rc:
        raise RuntimeError("fdmgpu_ns_info: %d" % rc)
    return torch.as_tensor(_DeviceField(ns, ptr.value, ns.shapes[name]), device="cuda")


class _Group(serve.Group):
    """A group whose end leaves no error code behind: it destroys an event it
    never made, which torch would report at its next call."""

    def close(self):
        super().close()
        hip.rt().hipGetLastError()


# ---- prepare and run --------------------------------------------------------
def prepare(case, seed):
    torch.zeros(1, device="cuda")   # torch's runtime first, then the library's
    kind = case["kind"]
    if kind == "ns":
        ns = fdm_amd.NSCube(nx=case["nx"], ny=case["ny"], nz=case["nz"], u0=NS_U0, Re=NS_RE, dt=NS_DT,
                            solver=case["prec"])
        for name, a in _ns_fields(case, seed).items():
            ns.set(name, a)
        return {"kind": kind, "ns": ns, "steps": case["steps"], "out": _Fields(ns, "uvwp")}
    rhs = _inputs(case, seed)
    if kind == "host":
        rhs = rhs.cpu().numpy().reshape(case["nz"], case["ny"], case["nx"])
        return {"kind": kind, "plan": _plan(case), "rhs": rhs, "ans": np.zeros_like(rhs)}
    ans = torch.zeros_like(rhs)
    shapes = _shapes(case)
    if kind in ("cube", "pcube", "rect"):
        dims = tuple(n for n in reversed(shapes[0]) if n)
        if case["batch"] > 1:
            dims = (case["batch"],) + dims
        return {"kind": "solve" if case["batch"] == 1 else "batch", "plan": _plan(case), "rhs": rhs.view(dims),
                "ans": ans.view(dims)}
    problems = [_problem(s, case["prec"], a, r)
                for s, a, r in zip(shapes, _views(ans, shapes), _views(rhs, shapes))]
    torch.cuda.synchronize()
    state = {"kind": kind, "rhs": rhs, "ans": ans, "problems": problems}
    if kind == "group":
        state["group"] = _Group(problems)
    else:
        state["server"] = serve.Server(8 << 30)
    return state


def run(state):
    kind = state["kind"]
    if kind == "solve":
        return state["plan"].solve(state["ans"], state["rhs"])
    if kind == "batch":
        return state["plan"].solve_batch(state["ans"], state["rhs"])
    if kind == "host":
        return state["plan"].solve(state["ans"], state["rhs"])
    if kind == "group":
        state["group"].solve(torch.cuda.current_stream().cuda_stream)
        return state["ans"]
    if kind == "serve":
        server = state["server"]
        tickets = [server.submit(p) for p in state["problems"]]
        for t in tickets:
            server.wait(t)
            server.forget(t)
        return state["ans"]
    state["ns"].step(state["steps"], torch.cuda.current_stream().cuda_stream)
    return state["out"]


# ---- what a pass cannot do without ------------------------------------------
def work(case):
    """Bytes: each right-hand side read once and each answer written once (a
    cavity step reads and writes u, v, w, p).  Flops: 5 N log2 N per complex
    N-point transform of two pencils, four or two transform passes per solve,
    about 8 per point for the tridiagonal systems; the cavity's stencils add
    about 120 per point."""
    es = 4 if case["prec"] == "f32" else 8

    def solve_flops(s):
        logs = [math.log2(n + 1) for n in s if n]
        t = logs[:2] if s[2] else logs[1:]
        return _points(s) * (2 * sum(2.5 * v for v in t) + 8)

    if case["kind"] == "ns":
        s = (case["nx"], case["ny"], case["nz"])
        return {"bytes": 64.0 * _points(s) * case["steps"],
                "flops": (solve_flops(s) + 120.0 * _points(s)) * case["steps"]}
    shapes = _shapes(case)
    return {"bytes": float(2 * es * sum(_points(s) for s in shapes)), "flops": sum(solve_flops(s) for s in shapes)}


# ---- the same answers in 64 bits, from torch alone --------------------------
def _sine(n):
    """The orthonormal sine matrix of n interior points (its own inverse)."""
    k = torch.arange(1, n + 1, dtype=torch.int64)
    m = (k[:, None] * k[None, :]) % (2 * (n + 1))
    return torch.sin(math.pi / (n + 1) * m.double()) * math.sqrt(2.0 / (n + 1))


def _lambda(n, h):
    k = torch.arange(1, n + 1, dtype=torch.float64)
    return 4.0 / (h * h) * torch.sin(k * math.pi / (2.0 * (n + 1))) ** 2


def _along(m, t, axis):
    """m applied along one axis of t (m symmetric)."""
    return torch.movedim(torch.tensordot(t, m, dims=([axis], [0])), -1, axis)


def _solve64(f, spacings, cache):
    """Dirichlet solve of the discrete Laplacian: sine transforms on every axis.
    f: [..., axes]; spacings in the order of the axes."""
    d = len(spacings)
    lead = f.dim() - d
    lam = None
    t = f
    for a, h in enumerate(spacings):
        n = f.shape[lead + a]
        if (n, h) not in cache:
            cache[(n, h)] = (_sine(n), _lambda(n, h))
        m, lm = cache[(n, h)]
        t = _along(m, t, lead + a)
        lm = lm.reshape([-1 if b == a else 1 for b in range(d)])
        lam = lm if lam is None else lam + lm
    t = t / -lam
    for a, h in enumerate(spacings):
        t = _along(cache[(f.shape[lead + a], h)][0], t, lead + a)
    return t


def _periodic64(f, spacings):
    lam = None
    for a, h in enumerate(spacings):
        n = f.shape[1 + a]
        k = torch.arange(n, dtype=torch.float64)
        lm = (4.0 / (h * h) * torch.sin(math.pi * k / n) ** 2).reshape([-1 if b == a else 1 for b in range(3)])
        lam = lm if lam is None else lam + lm
    lam[0, 0, 0] = 1.0
    c = torch.fft.fftn(f, dim=(1, 2, 3)) / -lam
    c[:, 0, 0, 0] = 0.0
    return torch.fft.ifftn(c, dim=(1, 2, 3)).real


def _ns64(case, seed):
    """The cavity's steps (the reference's staggered scheme, src/ns_cube.cpp:65-277)
    on whole arrays; index 0 of an axis holds its first ghost or face point."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    dx, dy, dz = PI2 / nx, PI2 / ny, PI2 / nz
    t = {k: torch.from_numpy(a).double() for k, a in _ns_fields(case, seed).items()}
    u, v, w, p = t["u"], t["v"], t["w"], t["p"]   # u x from -1, v y from -1, w z from -1
    cache = {}
    S = lambda a, n, o: slice(a + o, n + o + 1)   # noqa: E731  index range a..n at origin offset o

    def U(i, k, j):
        return u[S(*i, 0), S(*k, 0), S(*j, 1)]

    def V(i, k, j):
        return v[S(*i, 0), S(*k, 1), S(*j, 0)]

    def W(i, k, j):
        return w[S(*i, 1), S(*k, 0), S(*j, 0)]

    for _ in range(case["steps"]):
        # lid, ghost layers, pressure faces
        lim = min(nx + 1, nz + 1)
        u[nz + 1, :, 0:lim + 2] = 2 * NS_U0 - u[nz, :, 0:lim + 2]
        u[:, :, 0], u[:, :, nx + 2] = u[:, :, 2].clone(), u[:, :, nx].clone()
        v[:, 0, :], v[:, ny + 2, :] = v[:, 2, :].clone(), v[:, ny, :].clone()
        w[0], w[nz + 2] = w[2].clone(), w[nz].clone()
        I, K, J = slice(1, nz + 1), slice(1, ny + 1), slice(1, nx + 1)
        for q, n, h in ((0, nx, dx), (1, ny, dy), (2, nz, dz)):
            a = (u[I, K, :], v[I, :, J], w[:, K, J])[q]
            a = a.movedim((2, 1, 0)[q], 0)           # index 0 is -1
            b = p.movedim((2, 1, 0)[q], 0)
            inner = ((slice(None), I, K), (slice(None), I, J), (slice(None), K, J))[q]
            b = b[inner]
            b[0] = b[1] - (a[2] - 2 * a[1] + a[0]) / NS_RE / h
            b[n + 1] = b[n] - (a[n + 2] - 2 * a[n + 1] + a[n]) / NS_RE / h

        def diffuse(g, i, k, j):
            c = g(i, k, j)
            sh = lambda r, d: (r[0] + d, r[1] + d)   # noqa: E731
            return ((g(i, k, sh(j, 1)) - 2 * c + g(i, k, sh(j, -1))) / (NS_RE * dx * dx) +
                    (g(i, sh(k, 1), j) - 2 * c + g(i, sh(k, -1), j)) / (NS_RE * dy * dy) +
                    (g(sh(i, 1), k, j) - 2 * c + g(sh(i, -1), k, j)) / (NS_RE * dz * dz))

        def at(g, r, di, dk, dj):
            i, k, j = r
            return g((i[0] + di, i[1] + di), (k[0] + dk, k[1] + dk), (j[0] + dj, j[1] + dj))

        r = ((1, nz), (1, ny), (0, nx))
        F = at(U, r, 0, 0, 0) + NS_DT * (
            diffuse(U, *r) -
            ((0.5 * (at(U, r, 0, 0, 0) + at(U, r, 0, 0, 1))) ** 2 -
             (0.5 * (at(U, r, 0, 0, -1) + at(U, r, 0, 0, 0))) ** 2) / dx -
            0.25 * ((at(U, r, 0, 0, 0) + at(U, r, 0, 1, 0)) * (at(V, r, 0, 0, 1) + at(V, r, 0, 0, 0)) -
                    (at(U, r, 0, -1, 0) + at(U, r, 0, 0, 0)) * (at(V, r, 0, -1, 1) + at(V, r, 0, -1, 0))) / dy -
            0.25 * ((at(U, r, 0, 0, 0) + at(U, r, 1, 0, 0)) * (at(W, r, 0, 0, 1) + at(W, r, 0, 0, 0)) -
                    (at(U, r, -1, 0, 0) + at(U, r, 0, 0, 0)) * (at(W, r, -1, 0, 1) + at(W, r, -1, 0, 0))) / dz)
        r = ((1, nz), (0, ny), (1, nx))
        G = at(V, r, 0, 0, 0) + NS_DT * (
            diffuse(V, *r) -
            ((0.5 * (at(V, r, 0, 0, 0) + at(V, r, 0, 1, 0))) ** 2 -
             (0.5 * (at(V, r, 0, -1, 0) + at(V, r, 0, 0, 0))) ** 2) / dy -
            0.25 * ((at(U, r, 0, 0, 0) + at(U, r, 0, 1, 0)) * (at(V, r, 0, 0, 1) + at(V, r, 0, 0, 0)) -
                    (at(U, r, 0, 0, -1) + at(U, r, 0, 1, -1)) * (at(V, r, 0, 0, 0) + at(V, r, 0, 0, -1))) / dx -
            0.25 * ((at(W, r, 0, 0, 0) + at(W, r, 0, 1, 0)) * (at(V, r, 0, 0, 0) + at(V, r, 1, 0, 0)) -
                    (at(W, r, -1, 0, 0) + at(W, r, -1, 1, 0)) * (at(V, r, -1, 0, 0) + at(V, r, 0, 0, 0))) / dz)
        r = ((0, nz), (1, ny), (1, nx))
        H = at(W, r, 0, 0, 0) + NS_DT * (
            diffuse(W, *r) -
            ((0.5 * (at(W, r, 1, 0, 0) + at(W, r, 0, 0, 0))) ** 2 -
             (0.5 * (at(W, r, 0, 0, 0) + at(W, r, -1, 0, 0))) ** 2) / dz -
            0.25 * ((at(U, r, 1, 0, 0) + at(U, r, 0, 0, 0)) * (at(W, r, 0, 0, 1) + at(W, r, 0, 0, 0)) -
                    (at(U, r, 1, 0, -1) + at(U, r, 0, 0, -1)) * (at(W, r, 0, 0, 0) + at(W, r, 0, 0, -1))) / dx -
            0.25 * ((at(W, r, 0, 0, 0) + at(W, r, 0, 1, 0)) * (at(V, r, 0, 0, 0) + at(V, r, 1, 0, 0)) -
                    (at(W, r, 0, -1, 0) + at(W, r, 0, 0, 0)) * (at(V, r, 0, -1, 0) + at(V, r, 1, -1, 0))) / dy)
        rhs = ((F[:, :, 1:] - F[:, :, :-1]) / dx + (G[:, 1:] - G[:, :-1]) / dy + (H[1:] - H[:-1]) / dz) / NS_DT
        rhs[0] -= p[0, K, J] / dz ** 2
        rhs[-1] -= p[nz + 1, K, J] / dz ** 2
        rhs[:, 0] -= p[I, 0, J] / dy ** 2
        rhs[:, -1] -= p[I, ny + 1, J] / dy ** 2
        rhs[:, :, 0] -= p[I, K, 0] / dx ** 2
        rhs[:, :, -1] -= p[I, K, nx + 1] / dx ** 2
        x = _solve64(rhs, (dz, dy, dx), cache)
        u[I, K, 2:nx + 1] = F[:, :, 1:-1] - NS_DT / dx * (x[:, :, 1:] - x[:, :, :-1])
        v[I, 2:ny + 1, J] = G[:, 1:-1] - NS_DT / dy * (x[:, 1:] - x[:, :-1])
        w[2:nz + 1, K, J] = H[1:-1] - NS_DT / dz * (x[1:] - x[:-1])
        p[I, K, J] = x
    return {"u": u, "v": v, "w": w, "p": p}


def exact(case, seed):
    if case["kind"] == "ns":
        return _ns64(case, seed)
    shapes = _shapes(case)
    flat = _inputs(case, seed).cpu().double()
    cache, parts = {}, []
    if case["kind"] in ("group", "serve"):
        for s, f in zip(shapes, _views(flat, shapes)):
            dims = [n for n in reversed(s) if n]
            parts.append(_solve64(f.reshape(dims), [PI2 / n for n in dims], cache).reshape(-1))
        return torch.cat(parts)
    dims = [n for n in reversed(shapes[0]) if n]
    f = flat.reshape([case["batch"]] + dims)
    h = [PI2 / n for n in dims]
    if case["kind"] == "pcube":
        t = torch.cat([_periodic64(f[b:b + 1], h) for b in range(case["batch"])])
    else:
        t = torch.cat([_solve64(f[b:b + 1], h, cache) for b in range(case["batch"])])
    return t.reshape(dims if case["batch"] == 1 else [case["batch"]] + dims)
