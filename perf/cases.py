"""The work that users of the AMG-FCG library have it do, as measurable cases.

Each case is one call of a user's program through `bootcmatchg_amd`, on
operators and settings of the kinds the library is used with: constant
coefficient 2D/3D stencils (isotropic and anisotropic) and 3D diffusion with
log-normal cell coefficients, one AMG setup per operator or per call, one or
many right-hand sides, the FP64 drop-in and the reduced precisions of the
preconditioner, from grids where launches and latency count (32^3) to four
million rows, with odd sizes between.

`path` is what is called:
  spmv / residual / relax  one building block on a device-resident operator;
                           relax runs `sweeps` L1-Jacobi sweeps
  precond                  one application of the AMG preconditioner
  fcg                      a solve on a kept hierarchy
  dropin                   setup and solve, operator and b resident on the GPU
  solve                    the whole of solve(): host arrays in, x out
  multi                    `rhs` right-hand sides on one kept hierarchy
  serve                    `requests` requests through the serving loop over
                           the operators of `pool` (name:grid[:eps], ...)
"""
import ctypes
import functools
import math

import numpy as np
import torch

import bootcmatchg_amd as bc
from bootcmatchg_amd import operators as ops

# settings of the library's own drop-in runs; a case overrides what it names
DEFAULTS = dict(solver_type=0, max_hrc=1, conv_ratio=0.8, aggrsweeps=2, aggrtype=0,
                max_levels=39, cycle_type=0, coarse_solver=4, relax_type=4,
                relaxnumber_coarse=16, prerelax_sweeps=4, postrelax_sweeps=4, itnlim=2000,
                rtol=1e-8)
PRECISION = {"fp64": bc.PREC_FP64, "fp32": bc.PREC_FP32, "bf16": bc.PREC_BF16}
# 2D 5-point 256^2 and 1024^2 (two anisotropies), 3D 7-point 32^3 .. 128^3
# and one log-normal 64^3: the operators of a serving process
POOL = ("poisson2d:256,aniso2d:1024:0.01,poisson2d:1024,poisson3d:32,poisson3d:64,"
        "poisson3d:96,poisson3d:128,lognormal3d:64")


def listed():
    return [
        # a caller's own Krylov method on a small grid: one product per call
        dict(name="spmv_poisson3d_32", path="spmv", op="poisson3d", grid=32),
        # a smoother used on its own, variable coefficients, an odd grid
        dict(name="relax_lognormal3d_101", path="relax", op="lognormal3d", grid=101, sweeps=4),
        # the preconditioner inside a caller's own iteration, large operator
        dict(name="precond_poisson3d_160", path="precond", op="poisson3d", grid=160),
        # the small complete solve (looser tolerance), launches and latency
        dict(name="dropin_poisson3d_32", path="dropin", op="poisson3d", grid=32, rtol=1e-6),
        # the headline: setup and solve of 4.1 million unknowns in FP64
        dict(name="dropin_poisson3d_160", path="dropin", op="poisson3d", grid=160),
        # repeated solves on a kept hierarchy (a time step, a pressure solve), FP32 cycles
        dict(name="fcg_fp32_poisson3d_160", path="fcg", op="poisson3d", grid=160,
             precision="fp32"),
        # repeated solves, odd 2D anisotropic grid, W-cycle, BF16 coarse operators
        dict(name="fcg_bf16_aniso2d_1023_w", path="fcg", op="aniso2d", grid=1023, eps=0.01,
             precision="bf16", aggrsweeps=3, cycle_type=2),
        # heterogeneous medium: bootstrap composite of three hierarchies, FP64
        dict(name="dropin_bootstrap_lognormal3d_128", path="dropin", op="lognormal3d", grid=128,
             max_hrc=3, conv_ratio=0.5),
        # solve() as a library call of a CPU program: host arrays, odd grid
        dict(name="solve_host_lognormal3d_61", path="solve", op="lognormal3d", grid=61),
        # smoothed aggregation: denser coarse operators, general sparse products
        dict(name="dropin_smoothed_poisson3d_64", path="dropin", op="poisson3d", grid=64,
             aggrtype=1),
        # 32 right-hand sides (load cases, shots) on one 2D anisotropic operator
        dict(name="multi32_fp32_aniso2d_2048_w", path="multi", op="aniso2d", grid=2048, eps=0.01,
             precision="fp32", aggrsweeps=3, cycle_type=2, rhs=32),
        # a busy server: requests on eight cached operators
        dict(name="serve_fp32_pool8_32req", path="serve", pool=POOL, precision="fp32",
             requests=32, slots=16),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    path = rng.choice(["spmv", "residual", "relax", "precond", "fcg", "fcg", "dropin", "dropin",
                       "solve", "multi", "serve"])
    if path == "serve":
        pool = []
        for _ in range(rng.randint(2, 5)):
            op = rng.choice(["poisson2d", "aniso2d", "poisson3d", "lognormal3d"])
            rows = _log(rng, 3e4, 1e6)
            g = round(rows ** (1 / 2 if op.endswith("2d") else 1 / 3))
            pool.append("%s:%d%s" % (op, g, ":%.3g" % _log(rng, 0.005, 0.5)
                                     if op == "aniso2d" else ""))
        return dict(path=path, pool=",".join(pool), precision=rng.choice(["fp64", "fp32"]),
                    requests=rng.randint(6, 40), slots=rng.choice([4, 8, 16]))
    op = rng.choice(["poisson3d", "poisson3d", "aniso2d", "poisson2d", "lognormal3d",
                     "lognormal3d"])
    smoothed = path == "dropin" and op == "poisson3d" and rng.random() < 0.3
    lo, hi = {"spmv": (4e3, 4.19e6), "residual": (4e3, 4.19e6), "relax": (4e3, 4.19e6),
              "precond": (2e4, 4.19e6), "fcg": (2e4, 4.19e6), "dropin": (2e4, 4.19e6),
              "solve": (2e3, 6e5), "multi": (2e4, 4.19e6)}[path]
    if smoothed:
        lo, hi = 2e4, 3e5
    if op == "lognormal3d":
        hi = min(hi, 2.1e6)
    rows = _log(rng, lo, hi)
    d = dict(path=path, op=op, grid=round(rows ** (1 / 2 if op.endswith("2d") else 1 / 3)))
    if op == "aniso2d":
        d["eps"] = float("%.3g" % _log(rng, 0.005, 0.5))
    if path == "relax":
        d["sweeps"] = rng.randint(1, 6)
    if path in ("precond", "fcg", "dropin", "multi"):
        d["precision"] = rng.choice(["fp64", "fp64", "fp32", "bf16"])
    if smoothed:
        d.update(aggrtype=1, precision="fp64")
    elif path in ("precond", "fcg", "dropin", "solve", "multi"):
        d["cycle_type"] = rng.choice([0, 0, 1, 2]) if op.endswith("2d") else 0
        d["aggrsweeps"] = rng.choice([2, 3]) if op.endswith("2d") else 2
        if op == "lognormal3d" and path in ("fcg", "dropin") and rng.random() < 0.5:
            d.update(max_hrc=rng.choice([2, 3]), conv_ratio=0.5,
                     solver_type=rng.choice([0, 0, 1, 2]))
    if path == "multi":
        d["rhs"] = max(2, min(32, int(32 * 4.19e6 / rows), round(_log(rng, 2, 32))))
    return d


# ------------------------------------------------------------------ inputs

class _Dev:
    """A torch tensor passed to the library by its device address."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())


@functools.lru_cache(maxsize=None)
def _constant(op, grid, eps):
    if op == "poisson3d":
        return ops.poisson3d(grid)
    return ops.aniso2d(grid, eps)


def _operator(op, grid, eps, seed):
    if op == "lognormal3d":
        return ops.lognormal3d(grid, 4.0, seed=seed)
    return _constant(op, grid, 1.0 if op != "aniso2d" else eps)


def _case_operator(case, seed):
    return _operator(case["op"], case["grid"], case.get("eps", 1.0), seed)


def _uniform(seed, *shape):
    """Uniform[-1, 1) on the GPU from the seed."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.rand(*shape, dtype=torch.float64, device="cuda", generator=g) * 2.0 - 1.0


def _params(case):
    return bc.make_params(**{k: case.get(k, v) for k, v in DEFAULTS.items()})


def _abs_row_sums(A):
    return np.add.reduceat(np.abs(A[2]), A[0][:-1])


def _pool(case):
    out = []
    for item in case["pool"].split(","):
        p = item.split(":")
        out.append((p[0], int(p[1]), float(p[2]) if len(p) > 2 else 1.0))
    return out


def _requests(case, seed):
    """(operator index, seed of b) of each request: which operators are asked
    for belongs to the case, the right-hand sides to the seed."""
    n = len(_pool(case))
    r = np.random.default_rng(1000 * n + case["requests"])
    return [(int(r.integers(0, n)), seed * 1009 + k) for k in range(case["requests"])]


def prepare(case, seed):
    path = case["path"]
    s = {"case": case}
    if path == "solve":
        A = _case_operator(case, seed)
        s.update(A=A, prm=_params(case), b=ops.uniform_pm1(seed, len(A[0]) - 1))
        return s
    ctx = bc.Context(0)
    s["ctx"] = ctx
    prec = PRECISION[case.get("precision", "fp64")]
    if path == "serve":
        boots, sizes = [], []
        for op, grid, eps in _pool(case):
            A = _constant(op, grid, eps) if op != "lognormal3d" else _fixed_lognormal(grid)
            B = bc.Boot(ctx, bc.Csr(ctx, A), bc.make_params(**DEFAULTS))
            B.set_precision(prec)
            boots.append(B)
            sizes.append(len(A[0]) - 1)
        S = bc.Server(ctx, slots_per_operator=case["slots"])
        s.update(server=S, boots=boots, ids=[S.add(B) for B in boots])
        s["todo"] = []
        for op, bseed in _requests(case, seed):
            b = _uniform(bseed, sizes[op])
            s["todo"].append((op, _Dev(b), _Dev(torch.zeros_like(b))))
    else:
        A = _case_operator(case, seed)
        n = len(A[0]) - 1
        dA = bc.Csr(ctx, A)
        s.update(A=dA, prm=_params(case), prec=prec)
        if path == "multi":
            b = _uniform(seed, case["rhs"], n)
            x = torch.zeros_like(b)
            s.update(x=x, bs=[_Dev(b[j]) for j in range(case["rhs"])],
                     xs=[_Dev(x[j]) for j in range(case["rhs"])])
        else:
            s.update(b=_Dev(_uniform(seed, n)),
                     x=_Dev(_uniform(seed + 7919, n) if path in ("spmv", "residual", "relax")
                            else torch.zeros(n, dtype=torch.float64, device="cuda")))
        if path in ("spmv", "residual"):
            s["y"] = _Dev(torch.zeros(n, dtype=torch.float64, device="cuda"))
        if path == "relax":
            s["d"] = _Dev(torch.from_numpy(_abs_row_sums(A)).cuda())
            s["scratch"] = _Dev(torch.zeros(n, dtype=torch.float64, device="cuda"))
        if path in ("precond", "fcg", "multi"):
            s["B"] = bc.Boot(ctx, dA, s["prm"])
            s["B"].set_precision(prec)
    torch.cuda.synchronize()
    return s


@functools.lru_cache(maxsize=None)
def _fixed_lognormal(grid):
    return ops.lognormal3d(grid, 4.0, seed=0)


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "solve":
        x, info = bc.solve(s["A"], s["prm"], s["b"])
        return {"x": x, "iterations": info["iterations"]}
    ctx = s["ctx"]
    if path == "spmv":
        bc.spmv(ctx, s["A"], s["x"], s["y"])
        return {"y": s["y"].t}
    if path == "residual":
        bc.residual(ctx, s["A"], s["x"], s["b"], s["y"])
        return {"y": s["y"].t}
    if path == "relax":
        bc.relax(ctx, s["A"], s["d"], s["b"], s["x"], s["scratch"], case["sweeps"])
        return {"x": s["x"].t}
    if path == "precond":
        s["B"].precond(s["b"], s["x"])
        return {"x": s["x"].t}
    if path == "fcg":
        it, _ = s["B"].fcg(s["b"], s["x"])
        return {"x": s["x"].t, "iterations": it}
    if path == "dropin":
        B = bc.Boot(ctx, s["A"], s["prm"])
        if s["prec"]:
            B.set_precision(s["prec"])
        it, _ = B.fcg(s["b"], s["x"])
        B.free()
        return {"x": s["x"].t, "iterations": it}
    if path == "multi":
        it, _, _ = s["B"].fcg_multi(s["bs"], s["xs"])
        return {"x": s["x"], "iterations": it}
    # serve: two new requests between iterations until all are in
    S, todo, ids = s["server"], s["todo"], s["ids"]
    rids, done = [], 0
    while done < len(todo):
        for op, b, x in todo[len(rids):len(rids) + 2]:
            rids.append(S.submit(ids[op], b, x))
        done += S.step()
    res = [S.result(r) for r in rids]
    S.completed()
    return {"x": [x.t for _, _, x in todo],
            "iterations": np.array([r["iterations"] for r in res])}


# -------------------------------------------------- what a pass cannot avoid

def _size(op, grid):
    if op.endswith("2d"):
        n = grid * grid
        return n, 5 * n - 4 * grid
    n = grid ** 3
    return n, 7 * n - 6 * grid * grid


def _cycle_entries(case, nnz):
    """Matrix entries that one preconditioner application multiplies: per
    visit of a level the sweeps and the residual; level l has about
    nnz / 2^(aggrsweeps l) entries (more when smoothed: not counted)."""
    k = case.get("aggrsweeps", 2)
    visits = 1 + (case.get("cycle_type", 0) > 0)
    per = case.get("prerelax_sweeps", 4) + case.get("postrelax_sweeps", 4) + 1
    return nnz * per / (1.0 - visits / 2.0 ** k) * case.get("max_hrc", 1)


def work(case):
    """Bytes: the operator (values and columns), b and x once each. Flops: a
    product and a sum per multiplied entry; solves take a typical 30
    iterations of one cycle and one product each."""
    path = case["path"]
    if path == "serve":
        total = {"bytes": 0.0, "flops": 0.0}
        sizes = [_size(op, grid) for op, grid, _ in _pool(case)]
        share = case["requests"] / len(sizes)
        for n, nnz in sizes:
            total["bytes"] += 12.0 * nnz + 4.0 * n + 16.0 * n * share
            total["flops"] += 2.0 * 30 * share * (_cycle_entries({}, nnz) + nnz)
        return total
    n, nnz = _size(case["op"], case["grid"])
    matrix = 12.0 * nnz + 4.0 * n
    if path in ("spmv", "residual"):
        return {"bytes": matrix + (16.0 if path == "spmv" else 24.0) * n, "flops": 2.0 * nnz}
    if path == "relax":
        return {"bytes": matrix + 32.0 * n, "flops": 2.0 * nnz * case["sweeps"]}
    cyc = _cycle_entries(case, nnz)
    if path == "precond":
        return {"bytes": matrix + 24.0 * n, "flops": 2.0 * cyc}
    k = case.get("rhs", 1)
    return {"bytes": matrix + 16.0 * n * k, "flops": 2.0 * 30 * k * (cyc + nnz)}


# ------------------------------------------------------------ 64-bit answers

def _padded(A):
    """The CSR rows padded to the longest: columns (the row itself where
    there is no entry) and values (0 there), on the GPU."""
    row, col, val = (torch.from_numpy(np.asarray(a)).cuda() for a in A)
    row = row.long()
    n = row.numel() - 1
    length = row[1:] - row[:-1]
    K = int(length.max())
    k = torch.arange(K, device="cuda")
    have = k[None, :] < length[:, None]
    at = torch.where(have, row[:-1, None] + k[None, :], torch.zeros((), dtype=torch.long,
                                                                    device="cuda"))
    own = torch.arange(n, device="cuda")[:, None]
    cols = torch.where(have, col.long()[at], own)
    vals = torch.where(have, val[at], torch.zeros((), dtype=torch.float64, device="cuda"))
    return cols.t().contiguous(), vals.t().contiguous()


def _times(M, x):
    y = torch.zeros_like(x)
    for c, v in zip(*M):
        y += v * x[c]
    return y


def _cg(A, b):
    """Jacobi-preconditioned CG in 64 bits, far below the solver's tolerance."""
    M = _padded(A)
    n = b.numel()
    own = torch.arange(n, device="cuda")
    diag = torch.zeros_like(b)
    for c, v in zip(*M):
        diag += torch.where(c == own, v, torch.zeros_like(v))
    x = torch.zeros_like(b)
    r = b.clone()
    z = r / diag
    p = z.clone()
    rz = r @ z
    stop = 1e-12 * float(b.norm())
    for it in range(20000):
        q = _times(M, p)
        a = rz / (p @ q)
        x += a * p
        r -= a * q
        if it % 50 == 49 and float(r.norm()) <= stop:
            break
        z = r / diag
        new = r @ z
        p = z + (new / rz) * p
        rz = new
    return x


def _sine(x, axis):
    """DST-I along an axis (its own inverse times 2 / (N + 1))."""
    x = x.movedim(axis, -1)
    N = x.shape[-1]
    z = torch.zeros_like(x[..., :1])
    odd = torch.cat([z, x, z, -x.flip(-1)], dim=-1)
    return (-0.5 * torch.fft.rfft(odd).imag[..., 1:N + 1]).movedim(-1, axis)


def _sine_solve(op, grid, eps, b):
    """Direct solve of the constant-coefficient stencils by sine transforms."""
    k = torch.arange(1, grid + 1, dtype=torch.float64, device="cuda")
    lam = 4.0 * torch.sin(math.pi * k / (2 * (grid + 1))) ** 2
    scale = [1.0, 1.0, 1.0] if op == "poisson3d" else [eps, 1.0]
    d = len(scale)
    t = b.reshape([grid] * d)
    for a in range(d):
        t = _sine(t, a)
    ev = sum(s * lam.reshape([-1 if i == a else 1 for i in range(d)])
             for a, s in enumerate(scale))
    t = t / ev
    for a in range(d):
        t = _sine(t, a) * (2.0 / (grid + 1))
    return t.reshape(-1)


def _solution(op, grid, eps, A, b):
    if op == "lognormal3d":
        return _cg(A, b)
    return _sine_solve(op, grid, 1.0 if op != "aniso2d" else eps, b)


def exact(case, seed):
    path = case["path"]
    if path == "precond":
        return None
    if path == "serve":
        pool, xs = _pool(case), []
        for op, bseed in _requests(case, seed):
            name, grid, eps = pool[op]
            A = _fixed_lognormal(grid) if name == "lognormal3d" else None
            xs.append(_solution(name, grid, eps, A, _uniform(bseed, _size(name, grid)[0])))
        return {"x": xs, "iterations": None}
    op, grid, eps = case["op"], case["grid"], case.get("eps", 1.0)
    if path in ("spmv", "residual", "relax"):
        A = _case_operator(case, seed)
        n = len(A[0]) - 1
        M, b, x = _padded(A), _uniform(seed, n), _uniform(seed + 7919, n)
        if path == "spmv":
            return {"y": _times(M, x)}
        if path == "residual":
            return {"y": b - _times(M, x)}
        d = M[1].abs().sum(0)
        for _ in range(case["sweeps"]):
            x = x + (b - _times(M, x)) / d
        return {"x": x}
    A = _case_operator(case, seed) if op == "lognormal3d" else None
    n = _size(op, grid)[0]
    if path == "solve":
        b = torch.from_numpy(ops.uniform_pm1(seed, n)).cuda()
        return {"x": _solution(op, grid, eps, A, b).cpu().numpy(), "iterations": None}
    if path == "multi":
        b = _uniform(seed, case["rhs"], n)
        x = torch.empty_like(b)
        for j in range(case["rhs"]):
            x[j] = _solution(op, grid, eps, A, b[j])
        return {"x": x, "iterations": None}
    return {"x": _solution(op, grid, eps, A, _uniform(seed, n)), "iterations": None}
