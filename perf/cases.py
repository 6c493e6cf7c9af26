"""Cases that stand for what a program has this package do, through its public entry points.

Each case is a dict of plain values; ``prepare`` makes the inputs of a case on the GPU from a seed, ``run`` is one
pass, ``work`` the bytes and operations that a pass cannot do without and ``exact`` the same outputs in 64 bits from
plain numpy / torch.  Kinds:

* ``design``   a whole design iteration through a ``Network``: density filter, SIMP, stiffness, solve, compliance,
               and the adjoint back to dc/dx.  ``solver`` "default" is ``LinSolve`` without a solver (2D beams, the
               first thing a user runs); "fp32" / "fp64" are the multigrid CG of the 3D cantilever benchmark.
* ``solve``    one multigrid CG solve of one load on a new design (setup and solve, no network around it).
* ``loads``    several load cases of one projected (Heaviside) design as one block solve, Chebyshev smoother: the
               robust multi-load workload.
* ``heat``     a whole iteration on the scalar (conduction) matrix: assembly, solve, thermal compliance, gradient.
* ``product``  the fine-grid operator alone, K @ u and b - K u: what user-written iterations and checks call.
* ``chain``    density filter and SIMP forward, and both adjoints (``FilterConv`` radius and face conditions vary).
* ``sens``     the stiffness sensitivity alone: lambda^T dK/dx u per element.
* ``conv``     one convolution layer of the warm-start network: forward, gradient to the input, gradient to the
               weights (the layers differ in channels and grid).
* ``oc``       the optimality-criteria design update.

Sizes: the benchmark grids (120x40, 96x48x48, 128x64x64, 192x96x96, 256x128x128) and ragged ones like them.
"""
import math

import numpy as np
import torch

import pymoto_amd as pm
from pymoto_amd import _lib, problems

XMIN = 1e-9  # SIMP lower bound of every elasticity case


def listed():
    return [
        # the first script of a new user: the 2D half beam with the default solver; latency of many small launches
        {"name": "design-120x40", "kind": "design", "nx": 120, "ny": 40, "nz": 0, "solver": "default"},
        # the largest everyday grid, mixed precision: 12.8 million unknowns
        {"name": "design-256x128x128-fp32", "kind": "design", "nx": 256, "ny": 128, "nz": 128, "solver": "fp32"},
        # an ordinary 3D solve in full precision
        {"name": "solve-96x48x48-fp64", "kind": "solve", "nx": 96, "ny": 48, "nz": 48, "solver": "fp64"},
        # four load cases of one projected design, as the robust formulation has them
        {"name": "loads4-128x64x64", "kind": "loads", "nx": 128, "ny": 64, "nz": 64, "loads": 4, "solver": "fp32"},
        # heat conduction in a plate-like block
        {"name": "heat-80x80x48", "kind": "heat", "nx": 80, "ny": 80, "nz": 48},
        # the operator on a grid that divides by nothing
        {"name": "product-97x65x49", "kind": "product", "nx": 97, "ny": 65, "nz": 49},
        # filter and material law of the largest grid, the usual radius
        {"name": "chain-256x128x128-r1.5", "kind": "chain", "nx": 256, "ny": 128, "nz": 128, "radius": 1.5,
         "faces": "symmetric"},
        # a wide filter on a ragged grid
        {"name": "chain-75x51x33-r3.4", "kind": "chain", "nx": 75, "ny": 51, "nz": 33, "radius": 3.4, "faces": "edge"},
        # gradient of the 5.4 million unknown cantilever
        {"name": "sens-192x96x96", "kind": "sens", "nx": 192, "ny": 96, "nz": 96},
        # a full-resolution layer of the warm-start network at its training size
        {"name": "conv-128x64x64-16-16", "kind": "conv", "nx": 128, "ny": 64, "nz": 64, "cin": 16, "cout": 16},
        # a coarse layer of the same network
        {"name": "conv-32x16x16-64-64", "kind": "conv", "nx": 32, "ny": 16, "nz": 16, "cin": 64, "cout": 64},
        # the design update that follows every design iteration
        {"name": "oc-128x64x64", "kind": "oc", "nx": 128, "ny": 64, "nz": 64},
    ]


# ----------------------------------------------------------------------------------------------------------------
# drawn cases
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _levels_ok(nel):
    """Whether the multigrid hierarchy of the grid ends in a coarsest grid of an ordinary size."""
    nel = [n for n in nel if n]
    if any(n % 2 for n in nel):
        return False
    sub = [n // 2 for n in nel]
    while all(n % 2 == 0 for n in sub) and all(n >= 8 for n in sub):
        sub = [n // 2 for n in sub]
    return math.prod(n + 1 for n in sub) * len(sub) <= 3000


def _mg_grid(rng, lo, hi, most):
    """A 3D grid that coarsens at least twice, odd multiples of a power of two among its extents."""
    while True:
        p = 2 ** rng.randint(2, 5)
        nel = [p * max(1, round(_log(rng, lo, hi) / p)) for _ in range(3)]
        nel.sort(reverse=True)
        n = math.prod(v + 1 for v in nel)
        if min(nel) >= 8 and n <= most and n >= 2000 and _levels_ok(nel):
            return dict(zip(("nx", "ny", "nz"), nel))


def draw(rng):
    kind = rng.choice(["design", "design", "solve", "loads", "heat", "product", "chain", "chain", "sens", "conv", "conv",
                       "oc"])
    if kind == "design":
        if rng.random() < 0.5:
            while True:
                nx, ny = 4 * _log(rng, 8, 64), 4 * _log(rng, 5, 32)
                if _levels_ok((nx, ny)):
                    return {"kind": kind, "nx": nx, "ny": ny, "nz": 0, "solver": "default"}
        return {"kind": kind, **_mg_grid(rng, 16, 256, 4_300_000), "solver": rng.choice(["fp64", "fp32", "fp32"])}
    if kind == "solve":
        return {"kind": kind, **_mg_grid(rng, 16, 160, 700_000), "solver": rng.choice(["fp64", "fp32"])}
    if kind == "loads":
        k = rng.randint(2, 6)
        return {"kind": kind, **_mg_grid(rng, 16, 128, 2_000_000 // k), "loads": k, "solver": rng.choice(["fp64", "fp32"])}
    if kind == "heat":
        if rng.random() < 0.3:
            while True:
                nx, ny = 4 * _log(rng, 8, 96), 4 * _log(rng, 6, 64)
                if _levels_ok((nx, ny)):
                    return {"kind": kind, "nx": nx, "ny": ny, "nz": 0}
        return {"kind": kind, **_mg_grid(rng, 16, 128, 700_000)}
    if kind in ("product", "sens"):
        if rng.random() < 0.2:
            return {"kind": kind, "nx": _log(rng, 24, 900), "ny": _log(rng, 12, 500), "nz": 0}
        return {"kind": kind, "nx": _log(rng, 12, 256), "ny": _log(rng, 8, 128), "nz": _log(rng, 8, 128)}
    if kind == "chain":
        faces = rng.choice(["symmetric", "symmetric", "edge", "wrap", "constant"])
        if rng.random() < 0.25:
            return {"kind": kind, "nx": _log(rng, 30, 900), "ny": _log(rng, 20, 500), "nz": 0,
                    "radius": round(rng.uniform(1.2, 8.0), 1), "faces": faces}
        radius = round(rng.uniform(1.2, 4.6), 1)
        top = 256 if radius <= 3.0 else 96
        return {"kind": kind, "nx": _log(rng, 14, top), "ny": _log(rng, 12, top // 2), "nz": _log(rng, 12, top // 2),
                "radius": radius, "faces": faces}
    if kind == "conv":
        cin, cout = rng.choice([(8, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 32), (32, 16)])
        top = 128 if max(cin, cout) <= 16 else 64 if max(cin, cout) <= 32 else 32
        while True:
            nx, ny, nz = (4 * _log(rng, 2, max(2, t // 4)) for t in (top, top // 2, top // 2))
            if nx * ny * nz >= 512:
                return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "cin": cin, "cout": cout}
    if rng.random() < 0.3:
        return {"kind": "oc", "nx": _log(rng, 30, 400), "ny": _log(rng, 20, 200), "nz": 0}
    return {"kind": "oc", "nx": _log(rng, 16, 192), "ny": _log(rng, 8, 96), "nz": _log(rng, 8, 96)}


# ----------------------------------------------------------------------------------------------------------------
# inputs
def _nel(case):
    return tuple(n for n in (case["nx"], case["ny"], case["nz"]) if n)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rand(g, n, lo=0.0, hi=1.0):
    return lo + (hi - lo) * torch.rand(n, generator=g, dtype=torch.float64, device="cuda")


def _domain(case):
    return pm.VoxelDomain(case["nx"], case["ny"], case["nz"])


def _problem(d):
    bc, f = problems.cantilever3d(d) if d.dim == 3 else problems.mbb2d(d)
    return bc, torch.as_tensor(f, device="cuda")


def _smooth_density(g, nel, lo=0.0, hi=1.0):
    """A filtered random design: what SIMP and the solver meet (plain torch, the filter is not what is timed)."""
    x = _rand(g, math.prod(nel), lo, hi)
    return _filter64(x, nel, 1.5, "symmetric")


def _simp(x):
    return XMIN + (1.0 - XMIN) * x ** 3


def _project(x, beta=8.0, eta=0.5):
    a = math.tanh(beta * eta)
    return (a + torch.tanh(beta * (x - eta))) / (a + math.tanh(beta * (1.0 - eta)))


def _solver(d, precision, omega=0.5, tol=1e-10):
    levels = pm.solvers.auto_levels(d)
    mg = pm.solvers.build_hierarchy(d, levels, omega=omega, smooth_steps=2, precision=precision)
    return pm.solvers.CG(preconditioner=mg, tol=tol)


def _heat_problem(d):
    """Sink on the x = 0 side, uniform heat."""
    nj = np.arange(d.nely + 1)
    if d.dim == 3:
        jj, kk = np.meshgrid(nj, np.arange(d.nelz + 1), indexing="ij")
        bc = d.get_nodenumber(0, jj, kk).ravel()
    else:
        bc = d.get_nodenumber(0, nj)
    return np.sort(np.asarray(bc, dtype=np.int64)), torch.full((d.nnodes,), 1.0 / d.nnodes, dtype=torch.float64, device="cuda")


def _faces(case):
    v = 0.0 if case["faces"] == "constant" else case["faces"]
    return {a + "_bc": v for a in ("xmin", "xmax", "ymin", "ymax", "zmin", "zmax")}


def _design_x(case, seed):
    return _rand(_gen(seed), math.prod(_nel(case)))


def _oc_inputs(case, seed):
    g = _gen(seed)
    n = math.prod(_nel(case))
    x = 0.4 + 0.3 * (_rand(g, n) - 0.5)
    dg = -(0.05 + _rand(g, n)) ** 3  # compliance gradients: negative, over some orders of magnitude
    return x, dg


def _conv_inputs(case, seed):
    g = _gen(seed)
    n, ci, co = math.prod(_nel(case)), case["cin"], case["cout"]

    def normal(*shape):
        return torch.randn(*shape, generator=g, dtype=torch.float32, device="cuda")
    X = normal(n, ci).clamp_min_(0.0).to(torch.bfloat16)  # activations behind a ReLU
    W = (normal(27, co, ci) * math.sqrt(2.0 / (27 * ci))).to(torch.bfloat16)
    b = 0.1 * normal(co)
    dY = (1e-3 * normal(n, co)).to(torch.bfloat16)
    return X, W, b, dY


def _pair(case, seed):
    d = _domain(case)
    g = _gen(seed)
    n = d.dim * d.nnodes
    x = _simp(_smooth_density(g, _nel(case)))
    u, v = (torch.randn(n, generator=g, dtype=torch.float64, device="cuda") for _ in range(2))
    return d, x, u, v


def _loads_inputs(case, seed):
    d = _domain(case)
    g = _gen(seed)
    xs = _simp(_project(_smooth_density(g, _nel(case), 0.35, 1.0)))
    bc, _ = _problem(d)
    F = torch.as_tensor(problems.face_point_loads(d, case["loads"], int(seed) % 1000), device="cuda")
    return d, bc, xs, F


def prepare(case, seed):
    kind = case["kind"]
    if kind == "design":
        d = _domain(case)
        bc, f = _problem(d)
        x = _design_x(case, seed)
        sx = pm.Signal("x", x)
        if case["solver"] == "default":
            lin = pm.LinSolve(hermitian=True)
        else:
            lin = pm.LinSolve(hermitian=True, solver=_solver(d, case["solver"]))
        with pm.Network() as fn:
            sxf = pm.FilterConv(d, radius=1.5)(sx)
            ss = pm.MathExpression(f"{XMIN} + {1.0 - XMIN}*inp0^3")(sxf)
            sK = pm.AssembleStiffness(d, bc=bc)(ss)
            su = lin(sK, f)
            sc = pm.EinSum("i,i->")(su, f)
        return {"kind": kind, "fn": fn, "x": x, "sx": sx, "su": su, "sc": sc, "lin": lin}
    if kind == "solve":
        d = _domain(case)
        bc, f = _problem(d)
        xs = _simp(_smooth_density(_gen(seed), _nel(case)))
        return {"kind": kind, "assemble": pm.AssembleStiffness(d, bc=bc), "xs": xs, "f": f,
                "cg": _solver(d, case["solver"])}
    if kind == "loads":
        d, bc, xs, F = _loads_inputs(case, seed)
        return {"kind": kind, "assemble": pm.AssembleStiffness(d, bc=bc), "xs": xs, "f": F,
                "cg": _solver(d, case["solver"], omega="chebyshev")}
    if kind == "heat":
        d = _domain(case)
        bc, f = _heat_problem(d)
        sx = pm.Signal("x", _simp_heat(_smooth_density(_gen(seed), _nel(case))))
        lin = pm.LinSolve(hermitian=True, solver=_solver(d, "fp64"))
        with pm.Network() as fn:
            sK = pm.AssemblePoisson(d, bc=bc)(sx)
            su = lin(sK, f)
            sc = pm.EinSum("i,i->")(su, f)
        return {"kind": kind, "fn": fn, "sx": sx, "su": su, "sc": sc, "lin": lin}
    if kind == "product":
        d, x, u, v = _pair(case, seed)
        bc, _ = _problem(d)
        return {"kind": kind, "K": pm.AssembleStiffness(d, bc=bc)(x), "u": u, "b": v}
    if kind == "sens":
        d, x, u, v = _pair(case, seed)
        bc, _ = _problem(d)
        sx = pm.Signal("x", x)
        with pm.Network() as fn:
            sK = pm.AssembleStiffness(d, bc=bc)(sx)
        return {"kind": kind, "fn": fn, "sx": sx, "sK": sK, "u": u, "v": v}
    if kind == "chain":
        d = _domain(case)
        g = _gen(seed)
        sx = pm.Signal("x", _rand(g, d.nel))
        dy = torch.randn(d.nel, generator=g, dtype=torch.float64, device="cuda")
        with pm.Network() as fn:
            sxf = pm.FilterConv(d, radius=case["radius"], **_faces(case))(sx)
            ss = pm.MathExpression(f"{XMIN} + {1.0 - XMIN}*inp0^3")(sxf)
        return {"kind": kind, "fn": fn, "sx": sx, "ss": ss, "dy": dy}
    if kind == "conv":
        X, W, b, dY = _conv_inputs(case, seed)
        work = torch.empty(_lib.lib().pmt_conv3d_wgrad_work_size(case["cin"], case["cout"]), dtype=torch.float32,
                           device="cuda")
        return {"kind": kind, "X": X, "W": W, "b": b, "dY": dY, "Wt": torch.empty_like(W), "work": work,
                "dims": (case["nx"], case["ny"], case["nz"], case["cin"], case["cout"])}
    x, dg = _oc_inputs(case, seed)
    oc = pm.OC(pm.Signal("x", x), None, None, move=0.2, xmin=0.0, xmax=1.0, verbosity=0, maxvol=0.4)
    return {"kind": kind, "oc": oc, "x": x, "dg": dg}


def _simp_heat(x):
    return 1e-3 + (1.0 - 1e-3) * x ** 3


# ----------------------------------------------------------------------------------------------------------------
# one pass
def run(s):
    kind = s["kind"]
    if kind in ("design", "heat"):
        s["lin"].u = None  # the first iteration on this design: no earlier solution to start from
        s["fn"].reset()
        s["fn"].response()
        s["sc"].sensitivity = 1.0
        s["fn"].sensitivity()
        return {"c": s["sc"].state, "u": s["su"].state, "dcdx": s["sx"].sensitivity}
    if kind in ("solve", "loads"):
        s["cg"].update(s["assemble"](s["xs"]))
        return s["cg"].solve(s["f"])
    if kind == "product":
        return {"y": s["K"] @ s["u"], "r": s["K"].residual(s["b"], s["u"])}
    if kind == "sens":
        s["fn"].reset()
        s["fn"].response()
        s["sK"].sensitivity = pm.DyadicMatrix(s["v"], s["u"], fac=-1.0)
        s["fn"].sensitivity()
        return s["sx"].sensitivity
    if kind == "chain":
        s["fn"].reset()
        s["fn"].response()
        s["ss"].sensitivity = s["dy"]
        s["fn"].sensitivity()
        return {"y": s["ss"].state, "dx": s["sx"].sensitivity}
    if kind == "conv":
        lib, st, p = _lib.lib(), _lib.stream(), _lib.ptr
        *_, ci, co = s["dims"]
        n = s["X"].shape[0]
        out = {"Y": torch.empty(n, co, dtype=torch.bfloat16, device="cuda"),
               "dW": torch.empty(27, co, ci, dtype=torch.float32, device="cuda"),
               "db": torch.empty(co, dtype=torch.float32, device="cuda")}
        _lib.check(lib.pmt_conv3d_fwd(*s["dims"], p(s["X"]), p(s["W"]), p(s["b"]), 1, p(out["Y"]), st), "conv")
        _lib.check(lib.pmt_conv3d_bwd_weight(*s["dims"], p(s["X"]), p(s["dY"]), p(out["dW"]), p(out["db"]),
                                             p(s["work"]), st), "conv weight gradient")
        if ci >= 16:  # the network's first layer (8 channels) has no gradient to its input
            out["dX"] = torch.empty(n, ci, dtype=torch.bfloat16, device="cuda")
            _lib.check(lib.pmt_conv3d_bwd_data(*s["dims"], p(s["dY"]), p(s["W"]), p(s["Wt"]), p(out["dX"]), st),
                       "conv input gradient")
        return out
    return s["oc"].step(s["x"], s["dg"])


# ----------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
def work(case):
    kind = case["kind"]
    nel = _nel(case)
    dim = len(nel)
    e, nn = math.prod(nel), math.prod(n + 1 for n in nel)
    n = dim * nn
    ne = 2 ** dim * dim
    chain = {"bytes": 8.0 * 8 * e, "flops": 40.0 * e}

    def krylov(n, e, ne, cols, its, steps, prec):
        """CG iterations of a V(steps, steps) cycle: operator passes and vector updates, each operand once."""
        w = 4.0 if prec == "fp32" else 8.0
        cycle = (2 * steps) * (3 * n * w + e * w) * 8 / 7
        step = 2 * n * 8 + e * 8 + 6 * n * 8
        flops = (2 * steps * 8 / 7 + 1) * 2.0 * ne * 10 * e
        return {"bytes": cols * its * (cycle + step), "flops": cols * its * flops}
    if kind == "design":
        prec = "fp64" if case["solver"] == "default" else case["solver"]
        steps, its = (5, 18) if case["solver"] == "default" else (2, 20)
        k = krylov(n, e, ne, 1, its, steps, prec)
        return {"bytes": k["bytes"] + chain["bytes"] + 8.0 * (2 * n + e), "flops": k["flops"] + chain["flops"]}
    if kind == "solve":
        return krylov(n, e, ne, 1, 20, 2, case["solver"])
    if kind == "loads":
        return krylov(n, e, ne, case["loads"], 20, 2, case["solver"])
    if kind == "heat":
        return krylov(nn, e, 2 ** dim, 1, 16, 2, "fp64")
    if kind == "product":
        return {"bytes": 8.0 * (5 * n + 2 * e), "flops": 2 * 2.0 * ne * 10 * e}
    if kind == "sens":
        return {"bytes": 8.0 * (2 * n + e), "flops": 2.0 * ne * 12 * e}
    if kind == "chain":
        r = case["radius"]
        taps = math.prod(2 * min(m, int(r - 1e-10)) + 1 for m in nel)
        return {"bytes": 8.0 * 8 * e, "flops": 4.0 * taps * e}
    if kind == "conv":
        ci, co = case["cin"], case["cout"]
        dx = ci >= 16
        return {"bytes": 2.0 * e * ((2 + dx) * ci + (2 + dx) * co) + 27.0 * ci * co * 6,
                "flops": (2 + dx) * 2.0 * 27 * ci * co * e}
    return {"bytes": 8.0 * 3 * e, "flops": 30 * 8.0 * e}


# ----------------------------------------------------------------------------------------------------------------
# the same outputs in 64 bits
def _filter64(x, nel, radius, faces):
    """Normalised linear-hat convolution of an element field, padded at the faces."""
    half = [min(m, int(radius - 1e-10)) for m in nel]
    xp = x.reshape(*reversed(nel))
    for ax, (m, p) in enumerate(zip(nel, half)):
        dim = len(nel) - 1 - ax
        if faces == "constant":
            pad = [0, 0] * ax + [p, p]
            xp = torch.nn.functional.pad(xp, pad)
        else:
            idx = np.pad(np.arange(m), p, mode=faces)
            xp = xp.index_select(dim, torch.as_tensor(idx, device=x.device))
    grids = np.meshgrid(*[np.arange(-p, p + 1) for p in reversed(half)], indexing="ij")
    w = np.maximum(0.0, radius - np.sqrt(sum(g.astype(float) ** 2 for g in grids)))
    w /= w.sum()
    y = torch.zeros(tuple(reversed(nel)), dtype=x.dtype, device=x.device)
    for at in np.ndindex(*w.shape):
        if w[at] > 0.0:
            y = y + float(w[at]) * xp[tuple(slice(a, a + m) for a, m in zip(at, reversed(nel)))]
    return y.reshape(-1)


def _element(dim, scalar):
    """Element matrix of the unit square / cube: plane strain or 3D elasticity (E = 1, nu = 0.3), or conduction."""
    corners = [[1 if (a >> b) & 1 else -1 for b in range(dim)] for a in range(2 ** dim)]
    mu, lam = 1.0 / 2.6, 0.3 / (1.3 * 0.4)
    K = 0.0
    for q in corners:
        pos = np.array(q) / math.sqrt(3.0)
        dN = np.array([[np.prod([(1 + c[b] * pos[b]) / 2 if b != d else c[d] / 1.0 for b in range(dim)])
                        for c in corners] for d in range(dim)])  # on the unit element: d/dx = 2 d/dxi, (1 + c xi)/2
        if scalar:
            K = K + dN.T @ dN / 2 ** dim
            continue
        pairs = [(1, 2), (2, 0), (1, 0)] if dim == 3 else [(0, 1)]
        B = np.zeros((dim + len(pairs), dim * 2 ** dim))
        for a in range(2 ** dim):
            for d in range(dim):
                B[d, dim * a + d] = dN[d, a]
            for r, (i, j) in enumerate(pairs):
                B[dim + r, dim * a + i] = dN[j, a]
                B[dim + r, dim * a + j] = dN[i, a]
        D = np.diag([2 * mu] * dim + [mu] * len(pairs))
        D[:dim, :dim] += lam
        K = K + B.T @ D @ B / 2 ** dim
    return K


class _Operator:
    """K(x) with Dirichlet rows and columns dropped and max(K0) on their diagonal, element by element in torch."""

    def __init__(self, nel, bc, scalar=False):
        dim = len(nel)
        ndof = 1 if scalar else dim
        self.K0 = torch.as_tensor(_element(dim, scalar), device="cuda")
        idx = [torch.arange(m, device="cuda") for m in nel]
        g = torch.meshgrid(*reversed(idx), indexing="ij")  # (z, y, x): the element order
        base, stride = 0, 1
        strides = []
        for m, gi in zip(nel, reversed(g)):
            base = base + gi * stride
            strides.append(stride)
            stride *= m + 1
        corner = torch.as_tensor([sum(((a >> b) & 1) * strides[b] for b in range(dim)) for a in range(2 ** dim)],
                                 device="cuda")
        nodes = base.reshape(-1, 1) + corner
        self.conn = (nodes[:, :, None] * ndof + torch.arange(ndof, device="cuda")).reshape(nodes.shape[0], -1)
        self.n = stride * ndof
        self.free = torch.ones(self.n, dtype=torch.float64, device="cuda")
        self.free[torch.as_tensor(np.asarray(bc, dtype=np.int64), device="cuda")] = 0.0
        self.diag_bc = float(self.K0.max())

    def apply(self, x, u):
        w = (u * self.free)[self.conn] @ self.K0 * x[:, None]
        y = torch.zeros_like(u).index_add_(0, self.conn.reshape(-1), w.reshape(-1))
        return y * self.free + self.diag_bc * (1.0 - self.free) * u

    def diagonal(self, x):
        w = (x[:, None] * torch.diagonal(self.K0)).reshape(-1)
        y = torch.zeros_like(self.free).index_add_(0, self.conn.reshape(-1), w)
        return y * self.free + self.diag_bc * (1.0 - self.free)

    def sens(self, u, v):
        return ((u * self.free)[self.conn] @ self.K0 * (v * self.free)[self.conn]).sum(1)

    def solve(self, x, f):
        """Direct solution of small systems, Jacobi CG of ordinary ones, None for those that take too long."""
        if self.n <= 70_000 and (self.conn.shape[1] <= 8 or self.n <= 12_000):
            import scipy.sparse as sps
            import scipy.sparse.linalg as spl
            c, xh, fr = self.conn.cpu().numpy(), x.cpu().numpy(), self.free.cpu().numpy()
            K0 = self.K0.cpu().numpy()
            m = c.shape[1]
            val = (xh[:, None, None] * K0 * fr[c][:, :, None] * fr[c][:, None, :]).reshape(-1)
            A = sps.csc_matrix((val, (np.repeat(c, m, axis=1).reshape(-1), np.tile(c, (1, m)).reshape(-1))),
                               shape=(self.n, self.n)) + sps.diags(self.diag_bc * (1.0 - fr))
            lu = spl.splu(A.tocsc())
            fh = f.cpu().numpy()
            u = lu.solve(fh)
            u = u + lu.solve(fh - A @ u)  # one step of refinement
            return torch.as_tensor(u, device="cuda")
        if self.n > 900_000:
            return None
        dinv = 1.0 / self.diagonal(x)
        u = torch.zeros_like(f)
        bn = float(f.norm())
        for outer in range(3):  # restarts from the true residual
            r = f - self.apply(x, u)
            z = dinv * r
            p, rz = z.clone(), r @ z
            for it in range(3000):
                q = self.apply(x, p)
                alpha = rz / (p @ q)
                u += alpha * p
                r -= alpha * q
                z = dinv * r
                new = r @ z
                p = z + (new / rz) * p
                rz = new
                if it % 25 == 0 and float(r.norm()) <= 1e-13 * bn:
                    break
            if float((f - self.apply(x, u)).norm()) <= 1e-12 * bn:
                return u
        return None


def exact(case, seed):
    kind = case["kind"]
    nel = _nel(case)
    if kind in ("design", "solve", "loads", "product", "sens"):
        if kind in ("product", "sens"):
            d, x, u, v = _pair(case, seed)
            op = _Operator(nel, _problem(d)[0])
            if kind == "sens":
                return -op.sens(u, v)
            y = op.apply(x, u)
            return {"y": y, "r": v - y}
        if math.prod(m + 1 for m in nel) * len(nel) > 900_000 or (kind == "loads" and case["nx"] > 64):
            return None
        if kind == "loads":
            d, bc, xs, F = _loads_inputs(case, seed)
            op = _Operator(nel, bc)
            cols = [op.solve(xs, F[:, k].contiguous()) for k in range(F.shape[1])]
            return None if any(c is None for c in cols) else torch.stack(cols, dim=1)
        bc, f = _problem(_domain(case))
        op = _Operator(nel, bc)
        if kind == "solve":
            return op.solve(_simp(_smooth_density(_gen(seed), nel)), f)
        x = _design_x(case, seed).requires_grad_(True)
        xs = _simp(_filter64(x, nel, 1.5, "symmetric"))
        u = op.solve(xs.detach(), f)
        if u is None:
            return None
        (dx,) = torch.autograd.grad(xs, x, -op.sens(u, u))
        return {"c": np.float64(float(u @ f)), "u": u, "dcdx": dx}
    if kind == "heat":
        if math.prod(m + 1 for m in nel) > 900_000:
            return None
        bc, f = _heat_problem(_domain(case))
        op = _Operator(nel, bc, scalar=True)
        x = _simp_heat(_smooth_density(_gen(seed), nel))
        u = op.solve(x, f)
        return None if u is None else {"c": np.float64(float(u @ f)), "u": u, "dcdx": -op.sens(u, u)}
    if kind == "chain":
        g = _gen(seed)
        x = _rand(g, math.prod(nel)).requires_grad_(True)
        dy = torch.randn(math.prod(nel), generator=g, dtype=torch.float64, device="cuda")
        y = _simp(_filter64(x, nel, case["radius"], case["faces"]))
        (dx,) = torch.autograd.grad(y, x, dy)
        return {"y": y.detach(), "dx": dx}
    if kind == "conv":
        X, W, b, dY = (t.double() for t in _conv_inputs(case, seed))
        ci, co = case["cin"], case["cout"]
        shape = tuple(reversed(nel))

        def padded(t):
            return torch.nn.functional.pad(t.reshape(*shape, -1), (0, 0, 1, 1, 1, 1, 1, 1))

        def window(t, tap):
            at = (tap // 9, (tap // 3) % 3, tap % 3)
            return t[tuple(slice(a, a + m) for a, m in zip(at, shape))].reshape(-1, t.shape[-1])
        Xp, dYp = padded(X), padded(dY)
        Y = b + sum(window(Xp, t) @ W[t].T for t in range(27))
        out = {"Y": Y.clamp_min(0.0), "dW": torch.stack([dY.T @ window(Xp, t) for t in range(27)]), "db": dY.sum(0)}
        if ci >= 16:
            out["dX"] = sum(window(dYp, 26 - t) @ W[t] for t in range(27))
        return out
    x, dg = _oc_inputs(case, seed)
    lo, hi = (x - 0.2).clamp_min(0.0), (x + 0.2).clamp_max(1.0)
    l1, l2 = 0.0, 100000.0
    while l2 - l1 > 1e-4:
        mid = 0.5 * (l1 + l2)
        new = torch.minimum(torch.maximum(x * torch.sqrt(-dg / mid), lo), hi)
        l1, l2 = (mid, l2) if float(new.sum()) - 0.4 * x.numel() > 0 else (l1, mid)
    return new
