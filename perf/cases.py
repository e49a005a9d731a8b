"""The work this backend is measured on: solver programs over its public entry
points (ops_amd.ops, ops_amd.apps, ops_amd.serve), from calls of a few
microseconds of GPU work to grids that fill HBM bandwidth.

  laplace   the Laplace tutorial's Jacobi loop with its error read back every
            iteration: as the C++ application (host arrays in and out) and as
            loops on dats that stay on the GPU
  heat      a TeaLeaf implicit step in 2D or 3D: initial residual and a few
            CG iterations, FP64, variable coefficients
  mixed     one correction of the mixed-precision Poisson solver: FP64
            residual, a few FP32 preconditioned CG iterations, FP64 update
  adi       one ADI step: 7-point preprocessing, tridiagonal solves along x
            and y in place and along z accumulated into u (Thomas or PCR)
  trid      batched tridiagonal solves along one dimension after another
  serve     independent solves on the batched engine, submitted together and
            fetched as they complete
  halo      the halo exchange of a block-structured 2D grid

Outputs that live in dats come back as tensors over the dats' memory.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

from ops_amd import apps, ops, serve

# ------------------------------------------------------------------ the cases


def listed():
    return [
        # a small grid solved by the C++ application: the loop's latency
        {"name": "laplace_app_96x70", "path": "laplace", "app": True, "nx": 96, "ny": 70, "iters": 100},
        # the tutorial's own grid (4094 is not a multiple of any tile)
        {"name": "laplace_4094", "path": "laplace", "app": False, "nx": 4094, "ny": 4094, "iters": 20},
        # a middling 3D grid with odd sides: caches, tile remainders, latency
        {"name": "heat3d_197x150x131", "path": "heat", "ndim": 3, "nx": 197, "ny": 150, "nz": 131, "iters": 6},
        # the benchmark's grid
        {"name": "heat3d_512", "path": "heat", "ndim": 3, "nx": 512, "ny": 512, "nz": 512, "iters": 4},
        # TeaLeaf proper is two-dimensional
        {"name": "heat2d_3001x2003", "path": "heat", "ndim": 2, "nx": 3001, "ny": 2003, "nz": 1, "iters": 6},
        # FP32 inner iterations on a grid beyond the caches
        {"name": "mixed_400x384x390", "path": "mixed", "nx": 400, "ny": 384, "nz": 390, "iters": 8},
        # the benchmark's ADI grid, Thomas
        {"name": "adi_256", "path": "adi", "nx": 256, "ny": 256, "nz": 256, "pcr": False},
        # the ADI application's default solver, uneven sides
        {"name": "adi_pcr_200x130x97", "path": "adi", "nx": 200, "ny": 130, "nz": 97, "pcr": True},
        # single precision, odd row length
        {"name": "trid_f32_301x203x150", "path": "trid", "dtype": "f32", "nx": 301, "ny": 203, "nz": 150},
        # one small request: what a user waits for
        {"name": "serve_one_64", "path": "serve", "two": 1, "lo2": 64, "hi2": 64, "three": 0, "lo3": 0, "hi3": 0,
         "mixed": 0},
        # a batch of uneven 2D and 3D requests, one third of them with FP32 inner solves
        {"name": "serve_batch_12", "path": "serve", "two": 8, "lo2": 64, "hi2": 1000, "three": 4, "lo3": 32,
         "hi3": 128, "mixed": 3},
        # blocks of a multi-block program exchanging halos
        {"name": "halo_4x3_blocks", "path": "halo", "ngx": 4, "ngy": 3, "nx": 250, "ny": 181, "depth": 2, "comps": 1,
         "dtype": "f64"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["laplace", "heat", "heat", "mixed", "adi", "adi", "trid", "serve", "serve", "halo"])
    if path == "laplace":
        app = rng.random() < 0.5
        top = 600 if app else 4094
        return {"path": path, "app": app, "nx": _log(rng, 48, top), "ny": _log(rng, 48, top),
                "iters": 100 if app else 20}
    if path == "heat":
        if rng.random() < 0.4:
            return {"path": path, "ndim": 2, "nx": _log(rng, 64, 4000), "ny": _log(rng, 64, 4000), "nz": 1,
                    "iters": 6}
        return {"path": path, "ndim": 3, "nx": _log(rng, 24, 500), "ny": _log(rng, 24, 500), "nz": _log(rng, 24, 500),
                "iters": 4}
    if path == "mixed":
        return {"path": path, "nx": _log(rng, 32, 440), "ny": _log(rng, 32, 440), "nz": _log(rng, 32, 440),
                "iters": 8}
    if path == "adi":
        return {"path": path, "nx": _log(rng, 24, 300), "ny": _log(rng, 24, 300), "nz": _log(rng, 24, 300),
                "pcr": rng.random() < 0.5}
    if path == "trid":
        return {"path": path, "dtype": rng.choice(["f32", "f64"]), "nx": _log(rng, 24, 300), "ny": _log(rng, 24, 300),
                "nz": _log(rng, 24, 300)}
    if path == "serve":
        two, three = rng.randint(1, 6), rng.randint(0, 3)
        lo2, lo3 = _log(rng, 40, 300), _log(rng, 32, 64)
        return {"path": path, "two": two, "lo2": lo2, "hi2": lo2 + _log(rng, 8, 500), "three": three, "lo3": lo3,
                "hi3": lo3 + _log(rng, 4, 60), "mixed": rng.choice([0, 2, 3])}
    return {"path": "halo", "ngx": rng.randint(2, 4), "ngy": rng.randint(1, 4), "nx": _log(rng, 30, 1500),
            "ny": _log(rng, 30, 1500), "depth": rng.randint(1, 3), "comps": rng.choice([1, 1, 2]),
            "dtype": rng.choice(["f64", "f32"])}


# ------------------------------------------------------------------ dats as tensors
R, W, RW, INC, MAX = ops.OPS_READ, ops.OPS_WRITE, ops.OPS_RW, ops.OPS_INC, ops.OPS_MAX
_TYPE = {"f64": ("double", np.float64, "<f8", torch.float64), "f32": ("float", np.float32, "<f4", torch.float32)}


class Field:
    """A dat, freed when neither the program nor a tensor over its memory is
    left."""

    def __init__(self, block, size, name, dtype="f64", comps=1, depth=1):
        nd = len(size)
        self.type, npt, self.typestr, self.torch = _TYPE[dtype]
        self.dat = ops.ops_decl_dat(block, list(size), [-depth] * nd, [depth] * nd, npt, name, dim=comps)
        self.size, self.comps, self.depth = list(size), comps, depth

    def __del__(self):
        ops.ops_free_dat(self.dat)

    def arg(self, stencil, acc):
        return ops.ops_arg_dat(self.dat, self.comps, stencil, self.type, acc)

    def tensor(self, views, whole=False):
        """The dat's interior (or whole array) as it is in memory now, [z,]y,x[,component];
        views: the owner's cache (fused loop chains alternate two buffers)."""
        core = self.dat.core
        key = (core.data_d, whole)
        t = views.get(key)
        if t is None:
            t = views[key] = torch.as_tensor(_Memory(self, core, whole), device="cuda")
        return t

    def fill(self, values, whole=False):
        """values (a tensor of the interior's or the whole array's shape) into the dat"""
        space = C.c_int(ops.OPS_DEVICE)
        ops.lib().ops_dat_get_raw_pointer(self.dat.ptr, 0, None, C.byref(space))
        ops._check()
        self.tensor({}, whole).copy_(values)
        torch.cuda.synchronize()
        ops.lib().ops_dat_release_raw_data(self.dat.ptr, 0, W)
        ops._check()


class _Memory:
    def __init__(self, field, core, whole):
        self.field = field  # keeps the dat while a tensor is left
        nd, es = len(field.size), core.type_size
        h = field.depth if whole else 0
        pitch = [es * field.comps]
        for d in range(nd - 1):
            pitch.append(pitch[-1] * core.size[d])
        start = core.data_d + core.base_offset - h * sum(pitch)
        shape = [n + 2 * h for n in reversed(field.size)]
        strides = list(reversed(pitch))
        if field.comps > 1:
            shape.append(field.comps)
            strides.append(es)
        self.__cuda_array_interface__ = {"shape": tuple(shape), "strides": tuple(strides), "typestr": field.typestr,
                                         "data": (start, False), "version": 3}


class _Random:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))

    def uniform(self, shape):
        return torch.rand(shape, generator=self.gen, dtype=torch.float64, device="cuda")

    def normal(self, shape):
        return torch.randn(shape, generator=self.gen, dtype=torch.float64, device="cuda")


class State:
    pass


def _start():
    ops.ops_init(diags=0)


def _stencil(nd, pts, name, cache={}):  # noqa: B006 (stencils are declared once per process)
    key = (nd, tuple(pts))
    if key not in cache:
        cache[key] = ops.ops_decl_stencil(nd, len(pts) // nd, list(pts), name)
    return cache[key]


def _reduction(name, count=1, cache={}):  # noqa: B006
    if name not in cache:
        cache[name] = ops.ops_decl_reduction_handle(8 * count, "double", name)
    return cache[name]


def _block(nd, cache={}):  # noqa: B006
    if nd not in cache:
        cache[nd] = ops.ops_decl_block(nd, "grid%d" % nd)
    return cache[nd]


def _points(nd):
    """the point and the 5- or 7-point star, as flat offset lists"""
    point = [0] * nd
    star = list(point)
    for d in range(nd):
        for s in (-1, 1):
            star += [s if q == d else 0 for q in range(nd)]
    return point, star


def _gbl(v, type_="double"):
    return ops.ops_arg_gbl(v, 1, type_)


def _red(h, count=1, acc=INC):
    return ops.ops_arg_reduce(h, count, "double", acc)


# ------------------------------------------------------------------ laplace
def _laplace_init(case, seed):
    """the field with its boundary: a smooth top edge and a little noise"""
    nx, ny = case["nx"], case["ny"]
    rnd = _Random(seed)
    a = 0.1 * rnd.uniform((ny + 2, nx + 2))
    x = torch.arange(nx + 2, dtype=torch.float64, device="cuda")
    a[ny + 1] += torch.sin(math.pi * x / (nx + 1))
    return a


def _laplace_prepare(case, seed):
    s = State()
    init = _laplace_init(case, seed)
    if case["app"]:
        s.init = init.cpu().numpy()
        return s
    nx, ny = case["nx"], case["ny"]
    s.block = _block(2)
    point, star = _points(2)
    s0, s5 = _stencil(2, point, "point"), _stencil(2, star, "star")
    s.A, s.B, s.I = (Field(s.block, [nx, ny], n) for n in ("A", "Anew", "A0"))
    for f in (s.A, s.B, s.I):
        f.fill(init, whole=True)
    s.err = _reduction("error")
    s.apply = s.A.arg(s5, R), s.B.arg(s0, W)
    s.copy = s.A.arg(s0, W), s.B.arg(s0, R)
    s.reset = s.A.arg(s0, W), s.I.arg(s0, R)
    s.rng, s.views = [0, nx, 0, ny], {}
    return s


def _laplace_run(case, s):
    if case["app"]:
        err, hist, A = apps.laplace2d(case["nx"], case["ny"], case["iters"], 0, s.init)
        return {"A": A, "error": hist}
    hist = []
    ops.ops_par_loop("copy", "reset", s.block, 2, s.rng, *s.reset)
    for _ in range(case["iters"]):
        ops.ops_par_loop("apply_stencil", "apply_stencil", s.block, 2, s.rng, *s.apply, _red(s.err, 1, MAX))
        hist.append(float(ops.ops_reduction_result(s.err)))
        ops.ops_par_loop("copy", "copy", s.block, 2, s.rng, *s.copy)
    ops.ops_execute()
    return {"A": s.A.tensor(s.views), "error": np.array(hist)}


def _laplace_exact(case, seed):
    a = _laplace_init(case, seed)
    hist = []
    for _ in range(case["iters"]):
        b = 0.25 * (a[1:-1, 2:] + a[1:-1, :-2] + a[:-2, 1:-1] + a[2:, 1:-1])
        hist.append(float((b - a[1:-1, 1:-1]).abs().max()))
        a[1:-1, 1:-1] = b
    return {"A": a[1:-1, 1:-1].clone(), "error": np.array(hist)}


# ------------------------------------------------------------------ heat
def _heat_inputs(case, seed):
    """conductivity exp(N(0,1)) over the box with its halo, right-hand side
    U[0,1) plus a hot spot (the definitions of ops_amd/apps/problems.h)"""
    shape = [case["ny"], case["nx"]] if case["ndim"] == 2 else [case["nz"], case["ny"], case["nx"]]
    rnd = _Random(seed)
    K = torch.exp(rnd.normal([n + 2 for n in shape]))
    f = rnd.uniform(shape)
    sig = sum(shape) / 30.0
    g = torch.ones([1] * len(shape), dtype=torch.float64, device="cuda")
    for d, n in enumerate(shape):
        t = torch.arange(n, dtype=torch.float64, device="cuda") - 0.5 * (n - 1)
        g = g * torch.exp(-t * t / (2.0 * sig * sig)).reshape([-1 if q == d else 1 for q in range(len(shape))])
    f += 4.0 * g
    return K, f


def _heat_prepare(case, seed):
    nd = case["ndim"]
    n = [case["nx"], case["ny"], case["nz"]][:nd]
    s = State()
    s.block = _block(nd)
    point, star = _points(nd)
    unit = lambda d, v: [v if q == d else 0 for q in range(nd)]  # noqa: E731
    s0, sp = _stencil(nd, point, "point"), _stencil(nd, star, "star")
    sk = [_stencil(nd, point + unit(d, 1), "plus%d" % d) for d in range(nd)]
    sm = _stencil(nd, sum((unit(d, -1) for d in range(nd)), list(point)), "minus")
    names = ["Kx", "Ky", "Kz"][:nd]
    s.F = F = {k: Field(s.block, n, k) for k in ["u", "u0", "w", "r", "p"] + names}
    K, f = _heat_inputs(case, seed)
    F["p"].fill(K, whole=True)
    F["u0"].fill(f)
    del K, f
    full = sum(([-1, m + 1] for m in n), [])
    s.rng = sum(([0, m] for m in n), [])
    ext = sum(([0, m + 1] for m in n), [])
    a = lambda k, st, acc: F[k].arg(st, acc)  # noqa: E731
    loop = lambda k, r, *args: ops.ops_par_loop(k, k, s.block, nd, r, *args)  # noqa: E731
    loop("tea_leaf_recip_kernel", full, a("w", s0, W), a("p", s0, R))
    loop("tea_leaf_common_init_Kx_Ky_%skernel" % ("Kz_" if nd == 3 else ""), ext, *[a(k, s0, W) for k in names],
         a("w", sm, R))
    for d, k in enumerate(names):
        for lo, hi in ((-1, 1), (n[d], n[d] + 1)):
            r = list(full)
            r[2 * d:2 * d + 2] = [lo, hi]
            loop("tea_leaf_init_zero_kernel", r, a(k, s0, W))
    for k in ("w", "p"):
        loop("tea_leaf_init_zero_kernel", full, a(k, s0, W))
    ops.ops_mi_sync()
    s.red = _reduction("dot")
    rate = [_gbl(1.0) for _ in range(nd)]
    s.keep = rate
    kargs = [a(k, st, R) for k, st in zip(names, sk)]
    s.start = [a("u", s0, W), a("u0", s0, R)]
    s.init = [a("w", s0, W), a("r", s0, W), *kargs, a("u", sp, R)]
    s.first = [a("p", s0, W), a("r", s0, R)]
    s.dot = [a("r", s0, R), a("p", s0, R)]
    s.calc_w = [a("w", s0, W), *kargs, a("p", sp, R)]
    s.axpy = [a("u", s0, INC), a("p", s0, R)]
    s.ur = [a("r", s0, INC), a("w", s0, R)]
    s.axpby = [a("p", s0, RW), a("r", s0, R)]
    s.views = {k: {} for k in F}
    return s


def _heat_run(case, s):
    nd = case["ndim"]
    loop = lambda k, *args: ops.ops_par_loop(k + ("_3d" if nd == 3 and k in _3D else ""), k, s.block, nd, s.rng, *args)  # noqa: E731
    rate = [_gbl(1.0) for _ in range(nd)]
    loop("tea_leaf_yeqx_kernel", *s.start)
    loop("tea_leaf_common_init_kernel", *s.init, *rate)
    loop("tea_leaf_yeqx_kernel", *s.first)
    loop("tea_leaf_dot_kernel", *s.dot, _red(s.red))
    rro = float(ops.ops_reduction_result(s.red))
    hist = [rro]
    for _ in range(case["iters"]):
        loop("tea_leaf_cg_calc_w_reduce_kernel", *s.calc_w, *rate, _red(s.red))
        pw = float(ops.ops_reduction_result(s.red))
        alpha = _gbl(rro / pw)
        loop("tea_leaf_axpy_kernel", *s.axpy, alpha)
        loop("tea_leaf_cg_calc_ur_r_reduce_kernel", *s.ur, alpha, _red(s.red))
        rrn = float(ops.ops_reduction_result(s.red))
        loop("tea_leaf_axpby_kernel", *s.axpby, _gbl(rrn / rro), _gbl(1.0))
        hist += [pw, rrn]
        rro = rrn
    ops.ops_execute()
    return {**{k: s.F[k].tensor(s.views[k]) for k in ("u", "r", "p")}, "history": np.array(hist)}


_3D = ("tea_leaf_common_init_kernel", "tea_leaf_cg_calc_w_reduce_kernel")


def _heat_operator(K):
    """p -> A p of the TeaLeaf operator (unit rates) with zero flux through
    the faces; K over the box with its halo"""
    w = 1.0 / K
    nd = K.dim()
    faces = []
    for d in range(nd):
        mid = [slice(1, -1)] * nd
        hi, lo = list(mid), list(mid)
        hi[d], lo[d] = slice(1, None), slice(None, -1)
        a, b = w[tuple(lo)], w[tuple(hi)]
        k = (a + b) / (2.0 * a * b)  # n + 1 faces along d
        k.narrow(d, 0, 1).zero_()
        k.narrow(d, k.shape[d] - 1, 1).zero_()
        faces.append(k)
    del w

    def apply(p):
        out = p.clone()
        for d, k in enumerate(faces):
            n = p.shape[d]
            flux = k.narrow(d, 1, n - 1) * (p.narrow(d, 1, n - 1) - p.narrow(d, 0, n - 1))
            out.narrow(d, 0, n - 1).sub_(flux)
            out.narrow(d, 1, n - 1).add_(flux)
        return out

    return apply


def _heat_exact(case, seed):
    K, u = _heat_inputs(case, seed)
    A = _heat_operator(K)
    del K
    r = u - A(u)
    p = r.clone()
    rro = float((r * r).sum())
    hist = [rro]
    for _ in range(case["iters"]):
        w = A(p)
        pw = float((w * p).sum())
        u += (rro / pw) * p
        r -= (rro / pw) * w
        rrn = float((r * r).sum())
        p.mul_(rrn / rro).add_(r)
        hist += [pw, rrn]
        rro = rrn
    return {"u": u, "r": r, "p": p, "history": np.array(hist)}


# ------------------------------------------------------------------ mixed
def _mixed_prepare(case, seed):
    n = [case["nx"], case["ny"], case["nz"]]
    s = State()
    s.block = _block(3)
    point, star = _points(3)
    s0, sp = _stencil(3, point, "point"), _stencil(3, star, "star")
    s.F = F = {k: Field(s.block, n, k) for k in ("f", "x", "r")}
    F.update({k: Field(s.block, n, k, "f32") for k in ("e", "rr", "p", "w")})
    F["f"].fill(2.0 * _Random(seed).uniform(n[::-1]) - 1.0)
    s.rng = sum(([0, m] for m in n), [])
    s.red, s.dots = _reduction("dot"), _reduction("dots", 2)
    a = lambda k, st, acc: F[k].arg(st, acc)  # noqa: E731
    s.zero = [a("x", s0, W)]
    s.resid = [a("r", s0, W), a("f", s0, R), a("x", sp, R)]
    s.init = [a("e", s0, W), a("rr", s0, W), a("p", s0, W), a("r", s0, R)]
    s.calc_w = [a("w", s0, W), a("p", sp, R)]
    s.rr = [a("rr", s0, RW), a("w", s0, R)]
    s.e = [a("e", s0, RW), a("p", s0, R)]
    s.p = [a("p", s0, RW), a("rr", s0, R)]
    s.correct = [a("x", s0, RW), a("e", s0, R)]
    s.views = {k: {} for k in F}
    return s


def _mixed_run(case, s):
    loop = lambda k, *args: ops.ops_par_loop(k, k, s.block, 3, s.rng, *args)  # noqa: E731
    mi = _gbl(1.0 / 6.0, "float")
    loop("tea_leaf_init_zero_kernel", *s.zero)
    loop("poisson_residual_kernel", *s.resid, _red(s.red))
    hist = [float(ops.ops_reduction_result(s.red))]
    loop("mp_init_kernel", *s.init, mi, _red(s.dots, 2))
    rz = float(ops.ops_reduction_result(s.dots)[0])
    for _ in range(case["iters"]):
        loop("poisson_calc_w_reduce_kernel", *s.calc_w, _red(s.red))
        a = _gbl(rz / float(ops.ops_reduction_result(s.red)), "float")
        loop("mp_rr_update_kernel", *s.rr, a, mi, _red(s.dots, 2))
        loop("mp_e_update_kernel", *s.e, a)
        dots = ops.ops_reduction_result(s.dots)
        loop("mp_p_kernel", *s.p, mi, _gbl(float(dots[0]) / rz, "float"))
        rz = float(dots[0])
        hist += [rz, float(dots[1])]
    loop("mp_correct_kernel", *s.correct)
    ops.ops_execute()
    return {**{k: s.F[k].tensor(s.views[k]) for k in ("x", "rr", "p")}, "history": np.array(hist)}


def _poisson(p):
    out = 2.0 * p.dim() * p
    for d in range(p.dim()):
        n = p.shape[d]
        out.narrow(d, 1, n - 1).sub_(p.narrow(d, 0, n - 1))
        out.narrow(d, 0, n - 1).sub_(p.narrow(d, 1, n - 1))
    return out


def _mixed_exact(case, seed):
    r = 2.0 * _Random(seed).uniform([case["nz"], case["ny"], case["nx"]]) - 1.0
    x, p = torch.zeros_like(r), r / 6.0
    rz = float((r * r).sum())
    hist, rz = [rz], rz / 6.0
    for _ in range(case["iters"]):
        w = _poisson(p)
        a = rz / float((p * w).sum())
        x += a * p
        r -= a * w
        rr = float((r * r).sum())
        p = r / 6.0 + (rr / 6.0 / rz) * p
        rz = rr / 6.0
        hist += [rz, rr]
    return {"x": x, "rr": r, "p": p, "history": np.array(hist)}


# ------------------------------------------------------------------ adi
_COEF = ["ax", "bx", "cx", "ay", "by", "cy", "az", "bz", "cz"]


def _adi_input(case, seed):
    return _Random(seed).uniform([case["nz"], case["ny"], case["nx"]])


def _adi_prepare(case, seed):
    n = [case["nx"], case["ny"], case["nz"]]
    s = State()
    s.block = _block(3)
    point, star = _points(3)
    s0, sp = _stencil(3, point, "point"), _stencil(3, star, "star")
    s.F = F = {k: Field(s.block, n, k) for k in ["u", "du"] + _COEF}
    F["u"].fill(_adi_input(case, seed))
    for k, v in zip(("nx", "ny", "nz"), n):
        ops.ops_decl_const(k, 1, "int", v)
    ops.ops_decl_const("lambda", 1, "double", 1.0)
    s.rng = sum(([0, m] for m in n), [])
    s.pre = [F["u"].arg(sp, R)] + [F[k].arg(s0, W) for k in ["du"] + _COEF] + [ops.ops_arg_idx()]
    s.ctx = ops.TridParams(s.block, ops.TridParams.PCR if case["pcr"] else ops.TridParams.GATHER_SCATTER)
    s.out = {k: F[k].tensor({}) for k in ("u", "du")}
    return s


def _adi_run(case, s):
    F = s.F
    D = {k: f.dat for k, f in F.items()}
    ops.ops_par_loop("preproc_kernel", "preproc", s.block, 3, s.rng, *s.pre)
    ops.ops_tridMultiDimBatch(3, 0, s.rng, D["ax"], D["bx"], D["cx"], D["du"], s.ctx)
    ops.ops_tridMultiDimBatch(3, 1, s.rng, D["ay"], D["by"], D["cy"], D["du"], s.ctx)
    ops.ops_tridMultiDimBatch_Inc(3, 2, s.rng, D["az"], D["bz"], D["cz"], D["du"], D["u"], s.ctx)
    return s.out


def _thomas(a, b, c, d, dim):
    """tridiagonal solves along dimension dim of 64-bit tensors"""
    a, b, c, d = (t.movedim(dim, 0) for t in (a, b, c, d))
    n = d.shape[0]
    cp, dp = torch.empty_like(d), torch.empty_like(d)
    cp[0], dp[0] = c[0] / b[0], d[0] / b[0]
    for i in range(1, n):
        m = b[i] - a[i] * cp[i - 1]
        cp[i], dp[i] = c[i] / m, (d[i] - a[i] * dp[i - 1]) / m
    for i in range(n - 2, -1, -1):
        dp[i] -= cp[i] * dp[i + 1]
    return dp.movedim(0, dim)


def _adi_exact(case, seed):
    u = _adi_input(case, seed)
    inner = torch.zeros(u.shape, dtype=torch.bool, device="cuda")
    inner[1:-1, 1:-1, 1:-1] = True
    d = torch.zeros_like(u)
    d[1:-1, 1:-1, 1:-1] = -_poisson(u)[1:-1, 1:-1, 1:-1]
    off = torch.where(inner, -0.5, 0.0).double()
    b = torch.where(inner, 2.0, 1.0).double()
    for dim in (2, 1):
        d = _thomas(off, b, off, d, dim)
    return {"du": d, "u": u + _thomas(off, b, off, d, 0)}


# ------------------------------------------------------------------ trid
def _trid_inputs(case, seed):
    """diagonally dominant systems along each dimension, rounded to the dats' type"""
    rnd, shape, dt = _Random(seed), [case["nz"], case["ny"], case["nx"]], _TYPE[case["dtype"]][3]
    out = []
    for _ in range(3):
        a, c = rnd.uniform(shape) - 1.0, rnd.uniform(shape) - 1.0
        b = (a.abs() + c.abs()) + (0.1 + 0.9 * rnd.uniform(shape))
        out += [t.to(dt) for t in (a, b, c)]
    return out, (2.0 * rnd.uniform(shape) - 1.0).to(dt)


def _trid_prepare(case, seed):
    n = [case["nx"], case["ny"], case["nz"]]
    s = State()
    s.block = _block(3)
    s0 = _stencil(3, [0, 0, 0], "point")
    s.F = F = {k: Field(s.block, n, k, case["dtype"]) for k in ["d0", "d"] + _COEF}
    coef, d0 = _trid_inputs(case, seed)
    for k, v in zip(_COEF + ["d0"], coef + [d0]):
        F[k].fill(v)
    s.rng = sum(([0, m] for m in n), [])
    s.reset = [F["d"].arg(s0, W), F["d0"].arg(s0, R)]
    s.ctx = ops.TridParams(s.block)
    s.out = {"d": F["d"].tensor({})}
    return s


def _trid_run(case, s):
    F = s.F
    ops.ops_par_loop("copy", "copy", s.block, 3, s.rng, *s.reset)
    for d in range(3):
        a, b, c = (F[k].dat for k in _COEF[3 * d:3 * d + 3])
        ops.ops_tridMultiDimBatch(3, d, s.rng, a, b, c, F["d"].dat, s.ctx)
    return s.out


def _trid_exact(case, seed):
    coef, d = _trid_inputs(case, seed)
    d = d.double()
    for k in range(3):
        a, b, c = (t.double() for t in coef[3 * k:3 * k + 3])
        d = _thomas(a, b, c, d, 2 - k)
    return {"d": d}


# ------------------------------------------------------------------ serve
def _spread(count, lo, hi):
    """count sides from lo to hi, evenly spaced on a logarithmic scale"""
    return [int(round(lo * (hi / lo) ** (i / max(1, count - 1)))) for i in range(count)]


def _requests(case, seed):
    """(kind, side, mixed, seed) of each request; every mixed-th one has FP32 inner solves"""
    rnd = random.Random(int(seed))
    reqs = [(serve.POISSON2D, n) for n in _spread(case["two"], case["lo2"], case["hi2"])]
    reqs += [(serve.HEAT3D, n) for n in _spread(case["three"], case["lo3"], case["hi3"])]
    return [(k, n, bool(case["mixed"]) and i % case["mixed"] == 0, rnd.getrandbits(48)) for i, (k, n) in enumerate(reqs)]


_TOL = 1e-10


def _serve_prepare(case, seed):
    s = State()
    s.reqs = _requests(case, seed)
    s.server = _server()
    return s


def _server(cache={}):  # noqa: B006 (one engine serves the whole process)
    if not cache:
        cache[0] = serve.Server(budget_bytes=8 << 30, max_slots=64)
    return cache[0]


def _serve_run(case, s):
    ids = [s.server.submit(k, n, seed=q, tol=_TOL, mixed=m) for k, n, m, q in s.reqs]
    got = s.server.run()
    return [got[i][1] for i in ids]


def _mix64(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xbf58476d1ce4e5b9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94d049bb133111eb)
    return z ^ (z >> np.uint64(31))


def _u01(seed, stream, i):
    """the request inputs' generator (ops_amd/apps/problems.h), counters i"""
    G = np.uint64(0x9e3779b97f4a7c15)
    with np.errstate(over="ignore"):
        key = _mix64(np.array([seed], dtype=np.uint64) ^ (np.array([stream], dtype=np.uint64) * G))
        return (_mix64(key + (i + np.uint64(1)) * G) >> np.uint64(11)).astype(np.float64) * 2.0 ** -53


def _serve_exact(case, seed):
    out = []
    for kind, n, _, q in _requests(case, seed):
        if kind == serve.POISSON2D:
            f = torch.from_numpy(2.0 * _u01(q, 3, np.arange(n * n, dtype=np.uint64)) - 1.0).cuda().reshape(n, n)
            k = torch.arange(1, n + 1, dtype=torch.float64, device="cuda")
            S = torch.sin(math.pi * torch.outer(k, k) / (n + 1)) * math.sqrt(2.0 / (n + 1))
            lam = 4.0 * torch.sin(0.5 * math.pi * k / (n + 1)) ** 2
            out.append((S @ ((S @ f @ S) / (lam[:, None] + lam[None, :])) @ S).cpu().numpy())
            continue
        i = np.arange((n + 2) ** 3, dtype=np.uint64)
        a, b = _u01(q, 1, 2 * i), _u01(q, 1, 2 * i + np.uint64(1))
        K = np.exp(np.sqrt(-2.0 * np.log(1.0 - a)) * np.cos(2.0 * math.pi * b)).reshape(n + 2, n + 2, n + 2)
        t = np.arange(n) - 0.5 * (n - 1)
        g = np.exp(-t * t / (2.0 * (n / 10.0) ** 2))
        f = _u01(q, 2, np.arange(n ** 3, dtype=np.uint64)).reshape(n, n, n)
        f = f + 4.0 * g[:, None, None] * g[None, :, None] * g[None, None, :]
        A, u = _heat_operator(torch.from_numpy(K).cuda()), torch.from_numpy(f).cuda()
        r = u - A(u)
        p, rr = r.clone(), float((r * r).sum())
        stop = 1e-26 * rr
        while rr > stop:
            w = A(p)
            alpha = rr / float((p * w).sum())
            u += alpha * p
            r -= alpha * w
            new = float((r * r).sum())
            p.mul_(new / rr).add_(r)
            rr = new
        out.append(u.cpu().numpy())
    return out


# ------------------------------------------------------------------ halo
def _halo_inputs(case, seed):
    rnd, h = _Random(seed), case["depth"]
    shape = [case["ny"] + 2 * h, case["nx"] + 2 * h] + ([case["comps"]] if case["comps"] > 1 else [])
    return [rnd.uniform(shape).to(_TYPE[case["dtype"]][3]) for _ in range(case["ngx"] * case["ngy"])]


def _halo_pairs(case):
    """(from, to, iter_size, from_base, to_base) of every exchange between neighbours"""
    nx, ny, h, gx = case["nx"], case["ny"], case["depth"], case["ngx"]
    for j in range(case["ngy"]):
        for i in range(gx):
            b = i + gx * j
            if i > 0:
                yield b - 1, b, [h, ny], [nx - h, 0], [-h, 0]
                yield b, b - 1, [h, ny], [0, 0], [nx, 0]
            if j > 0:
                yield b - gx, b, [nx, h], [0, ny - h], [0, -h]
                yield b, b - gx, [nx, h], [0, 0], [0, ny]


def _halo_prepare(case, seed):
    s = State()
    s.u = []
    for v in _halo_inputs(case, seed):
        s.u.append(Field(_block(2), [case["nx"], case["ny"]], "u", case["dtype"], case["comps"], case["depth"]))
        s.u[-1].fill(v, whole=True)
    s.group = ops.ops_decl_halo_group([ops.ops_decl_halo(s.u[f].dat, s.u[t].dat, it, fb, tb, [1, 2], [1, 2])
                                       for f, t, it, fb, tb in _halo_pairs(case)])
    s.out = [f.tensor({}, whole=True) for f in s.u]
    return s


def _halo_run(case, s):
    ops.ops_halo_transfer(s.group)
    return s.out


def _halo_exact(case, seed):
    u, h = [t.double() for t in _halo_inputs(case, seed)], case["depth"]
    for f, t, it, fb, tb in _halo_pairs(case):
        box = [[slice(b[q] + h, b[q] + h + it[q]) for q in (1, 0)] for b in (fb, tb)]
        u[t][tuple(box[1])] = u[f][tuple(box[0])]
    return u


# ------------------------------------------------------------------ what is asked for
def prepare(case, seed):
    _start()
    s = globals()["_%s_prepare" % case["path"]](case, seed)
    s.case = dict(case)
    return s


def run(state):
    return globals()["_%s_run" % state.case["path"]](state.case, state)


def exact(case, seed):
    return globals()["_%s_exact" % case["path"]](case, seed)


def work(case):
    """Bytes: each pass between two reductions whose result the program needs
    reads its inputs and writes its outputs once.  Operations: those of the
    kernels as written."""
    k = case["path"]
    if k == "halo":
        es = {"f64": 8, "f32": 4}[case["dtype"]] * case["comps"]
        n = sum(it[0] * it[1] for _, _, it, _, _ in _halo_pairs(case))
        return {"bytes": 2.0 * n * es, "flops": 0.0}
    if k == "serve":
        by = fl = 0.0
        for kind, n, mixed, _ in _requests(case, 0):
            # CG iterations to 1e-10, about 3.3 n for the 2D Poisson problem and
            # 120 for the heat problem; 72 and 96 bytes a point and iteration
            # (half of that in FP32)
            pts, it, b, f = (n * n, 3.3 * n, 72.0, 16.0) if kind == serve.POISSON2D else (n ** 3, 120.0, 96.0, 36.0)
            by += pts * it * b * (0.5 if mixed else 1.0)
            fl += pts * it * f
        return {"bytes": by, "flops": fl}
    pts = float(case["nx"]) * case["ny"] * case.get("nz", 1)
    if k == "laplace":
        return {"bytes": pts * 24.0 * case["iters"], "flops": pts * 6.0 * case["iters"]}
    if k == "heat":
        coef = 8.0 * case["ndim"]
        # init: u0, K in; u, r, p, w out.  iteration: u, p, r, K in and u, p, w out; r, w in and r out
        return {"bytes": pts * (40.0 + coef + case["iters"] * (72.0 + coef)),
                "flops": pts * (case["iters"] + 1) * (9.0 + 9.0 * case["ndim"])}
    if k == "mixed":
        # f in, e, rr, p, x out; iteration: e, p, rr in and e, p, w out; rr, w in and rr out; x, e in, x out
        return {"bytes": pts * (28.0 + 36.0 * case["iters"] + 20.0), "flops": pts * 20.0 * case["iters"]}
    if k == "adi":
        return {"bytes": pts * (88.0 + 40.0 + 40.0 + 48.0), "flops": pts * 50.0}
    es = {"f64": 8.0, "f32": 4.0}[case["dtype"]]
    return {"bytes": pts * es * (2.0 + 15.0), "flops": pts * 36.0}


def tolerance(case):
    k = case["path"]
    if k in ("halo", "laplace"):
        return "exact"  # copies; an average, a difference and a maximum in a fixed order
    if k == "mixed":
        return {"rel": 5e-6}  # FP32 fields
    if k == "serve":
        return {"rel": 1e-8}  # solved to a relative residual of 1e-10
    if k == "trid":
        return {"rel": 1e-5 if case["dtype"] == "f32" else 1e-13}
    return {"rel": 1e-12}  # FP64 sums in another order, a few CG iterations on; PCR against Thomas
