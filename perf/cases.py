"""The work whose speed is watched: sparse products, smoothing steps, grid
transfers, Krylov and multigrid solves and batched solves, each through the
public binding (honei_amd), with device memory held by torch.

Every system is a Q1 discretisation on a (side x side) grid, as in the
framework's tests and benchmark, or a random banded ELL matrix with rows of
1..27 entries.  Inputs are made from the seed alone.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import honei_amd as H

DEV = "cuda"
VT = {"f32": H.F32, "f64": H.F64, "bf16": H.BF16}
TORCH = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.float32}   # vectors
VALUES = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16}  # stored values
SIZE = {"f32": 4, "f64": 8, "bf16": 2}
WIDTH, BAND = 27, 4096   # random matrices: entries per row at most, columns within +-BAND


def listed():
    return [
        # One step of a stand-alone Jacobi iteration on a small grid: sweep,
        # defect and its norm on the host, launch and return latency.
        {"name": "smooth_33_f64", "kind": "smooth", "side": 33, "dtype": "f64", "threads": 1, "host_norm": True},
        # The same step on a large grid with the norm left on the device.
        {"name": "smooth_1025_f32", "kind": "smooth", "side": 1025, "dtype": "f32", "threads": 1, "host_norm": False},
        # y = A x with the largest finite-element operator, double precision.
        {"name": "product_2049_f64", "kind": "product", "side": 2049, "dtype": "f64", "threads": 1},
        # y = A x of an irregular matrix in the plain ELL layout, odd size.
        {"name": "random_1000003_f32", "kind": "random", "n": 1000003, "dtype": "f32"},
        # y = A x of an irregular matrix through its sliced copy, double.
        {"name": "sliced_2000003_f64", "kind": "sliced", "n": 2000003, "dtype": "f64"},
        # Down and up one grid level, as a user's own multigrid cycle does.
        {"name": "transfer_1025_f32", "kind": "transfer", "level": 10, "dtype": "f32"},
        # Plain CG on a small system: hundreds of short dependent iterations.
        {"name": "cg_129_f64", "kind": "cg", "side": 129},
        # Jacobi-preconditioned CG on a jumping coefficient, ordinary size.
        {"name": "pcg_jacobi_385_f64", "kind": "pcg", "side": 385},
        # One large constant-coefficient problem by mixed-precision multigrid.
        {"name": "mixed_2049_f32", "kind": "mixed", "level": 11, "inner": "f32"},
        # One ordinary variable-coefficient problem by multigrid-CG.
        {"name": "mgcg_257_f32", "kind": "mgcg", "level": 8, "inner": "f32"},
        # A handful of systems at a time, 16-bit stored coarse operators.
        {"name": "batch_16_bf16", "kind": "batch", "inner": "bf16", "n5": 5, "n6": 4, "n7": 4, "n8": 3, "n9": 0},
        # The throughput workload: 256 systems of five sizes in one batch.
        {"name": "batch_256_f32", "kind": "batch", "inner": "f32", "n5": 61, "n6": 47, "n7": 44, "n8": 53, "n9": 51},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["smooth", "product", "random", "sliced", "transfer", "cg", "pcg", "mixed", "mgcg", "batch"])
    if kind == "smooth":
        return {"kind": kind, "side": _log(rng, 17, 1300), "dtype": rng.choice(["f32", "f64"]),
                "threads": rng.choice([1, 1, 2, 4]), "host_norm": rng.random() < 0.5}
    if kind == "product":
        return {"kind": kind, "side": _log(rng, 33, 2049), "dtype": rng.choice(["f32", "f64", "bf16"]),
                "threads": rng.choice([1, 1, 2, 4])}
    if kind in ("random", "sliced"):
        return {"kind": kind, "n": _log(rng, 9001, 2000003), "dtype": rng.choice(["f32", "f64"])}
    if kind == "transfer":
        return {"kind": kind, "level": rng.randint(4, 11), "dtype": rng.choice(["f32", "f64"])}
    if kind == "cg":
        return {"kind": kind, "side": _log(rng, 17, 300)}
    if kind == "pcg":
        return {"kind": kind, "side": _log(rng, 33, 385)}
    if kind == "mixed":
        return {"kind": kind, "level": rng.randint(5, 11), "inner": rng.choice(["f32", "f32", "bf16"])}
    if kind == "mgcg":
        return {"kind": kind, "level": rng.randint(5, 10), "inner": rng.choice(["f32", "f64", "bf16"])}
    return {"kind": kind, "inner": rng.choice(["f32", "f32", "bf16", "f64"]), "n5": _log(rng, 2, 60),
            "n6": _log(rng, 1, 45), "n7": _log(rng, 1, 44), "n8": _log(rng, 1, 40), "n9": rng.randint(0, 20)}


# ---- inputs ------------------------------------------------------------------
class Vec:
    """A torch tensor's memory as the binding takes it."""

    def __init__(self, t):
        self.t, self.ptr, self.n = t, t.data_ptr(), t.numel()


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _uniform(g, n, dtype=torch.float64):
    return torch.rand(n, generator=g, device=DEV, dtype=torch.float64).mul_(2).sub_(1).to(dtype)


def _lognormal(g, cells):
    return torch.exp(torch.randn(cells * cells, generator=g, device=DEV, dtype=torch.float64))


def _matrix(rows, stride, ncpr, threads, dtype, Aj, Ax, Arl):
    D = H.DeviceEll.__new__(H.DeviceEll)
    D.rows = D.cols = rows
    D.stride, D.ncpr, D.threads, D.vtype = stride, ncpr, threads, VT[dtype]
    D.Aj, D.Ax, D.Arl = Vec(Aj), Vec(Ax), Vec(Arl)
    return D


def _q1(side, dtype, threads=1, omega=0.8, coeff=None):
    """Q1 operator with Dirichlet identity rows and omega / diagonal."""
    n, ncpr = side * side, -(-9 // threads)
    stride = 32 * (-(-n * threads // 32))
    Aj = torch.zeros(ncpr * stride, dtype=torch.int32, device=DEV)
    Ax = torch.zeros(ncpr * stride, dtype=VALUES[dtype], device=DEV)
    Arl = torch.zeros(n, dtype=torch.int32, device=DEV)
    dinv = torch.empty(n, dtype=TORCH[dtype], device=DEV)
    H.call("honei_hip_q1_assemble", VT[dtype], side, Aj.data_ptr(), Ax.data_ptr(), Arl.data_ptr(), stride,
           None if coeff is None else coeff.data_ptr(), dinv.data_ptr(), omega, threads, None)
    return _matrix(n, stride, ncpr, threads, dtype, Aj, Ax, Arl), dinv


def _drop_boundary_columns(D, side):
    """Symmetric form of a threads = 1 operator: no couplings to the boundary."""
    Aj, Ax = D.Aj.t.view(D.ncpr, D.stride), D.Ax.t.view(D.ncpr, D.stride)
    r, c = Aj // side, Aj % side
    edge = (r == 0) | (r == side - 1) | (c == 0) | (c == side - 1)
    row = torch.arange(D.stride, device=DEV, dtype=torch.int32)
    Ax.masked_fill_(edge & (Aj != row), 0)


def _random_arrays(case, seed):
    """Aj, Ax [WIDTH][stride], Arl, x: rows of 1..WIDTH distinct ascending
    columns spread over the band, as the random product benchmark has them."""
    g, n, dt = _gen(seed), case["n"], TORCH[case["dtype"]]
    stride = 32 * (-(-n // 32))
    step = 2 * BAND // WIDTH
    k = torch.arange(WIDTH, device=DEV).view(WIDTH, 1)
    cols = torch.randint(0, step, (WIDTH, n), generator=g, device=DEV, dtype=torch.int32) + (k * step - BAND).int()
    cols += torch.arange(n, device=DEV, dtype=torch.int32)
    rank = torch.rand(WIDTH, n, generator=g, device=DEV).argsort(0).to(torch.int32)
    length = torch.randint(1, WIDTH + 1, (n,), generator=g, device=DEV, dtype=torch.int32)
    keep = (rank < length) & (cols >= 0) & (cols < n)
    order = (~keep).to(torch.int8).sort(stable=True, dim=0).indices
    arl = keep.sum(0).to(torch.int32)
    used = k < arl
    Aj = torch.zeros(WIDTH, stride, dtype=torch.int32, device=DEV)
    Ax = torch.zeros(WIDTH, stride, dtype=dt, device=DEV)
    Aj[:, :n] = torch.where(used, cols.gather(0, order), 0)
    Ax[:, :n] = torch.where(used, torch.randn(WIDTH, n, generator=g, device=DEV, dtype=dt), 0)
    return Aj, Ax, arl, _uniform(g, n, dt)


def _vectors(case, seed):
    """The vectors of a grid case: what prepare and exact share."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("smooth", "product"):
        dt, n = TORCH[case["dtype"]], case["side"] ** 2
        return _uniform(g, n, dt), _uniform(g, n, dt)
    if kind == "transfer":
        dt = TORCH[case["dtype"]]
        return (_uniform(g, (2 ** case["level"] + 1) ** 2, dt), _uniform(g, (2 ** (case["level"] - 1) + 1) ** 2, dt))
    if kind == "cg":   # homogeneous Dirichlet problem: no load on the boundary
        side = case["side"]
        return _uniform(g, side * side).view(side, side).masked_fill_(_edge(side), 0).view(-1)
    if kind == "pcg":
        return _lognormal(g, case["side"] - 1), _uniform(g, case["side"] ** 2)
    if kind == "mixed":
        return _uniform(g, (2 ** case["level"] + 1) ** 2)
    if kind == "mgcg":
        return _lognormal(g, 2 ** case["level"]), _uniform(g, (2 ** case["level"] + 1) ** 2)
    out = []
    for level in range(9, 4, -1):
        for _ in range(case["n%d" % level]):
            out.append((level, _lognormal(g, 2 ** level), _uniform(g, (2 ** level + 1) ** 2)))
    return out


def prepare(case, seed):
    H.init(0)
    kind, s = case["kind"], {"case": case}
    if kind in ("random", "sliced"):
        Aj, Ax, Arl, x = _random_arrays(case, seed)
        D = _matrix(case["n"], Aj.shape[1], WIDTH, 1, case["dtype"], Aj.view(-1), Ax.view(-1), Arl)
        s.update(D=D, x=Vec(x), y=Vec(torch.empty_like(x)))
        if kind == "sliced":
            torch.cuda.synchronize()
            s["S"] = H.Sell(D)
    elif kind == "product":
        x, _ = _vectors(case, seed)
        D, _ = _q1(case["side"], case["dtype"], case["threads"])
        s.update(D=D, x=Vec(x), y=Vec(torch.empty_like(x)))
    elif kind == "smooth":
        x, b = _vectors(case, seed)
        D, dinv = _q1(case["side"], case["dtype"], case["threads"])
        s.update(D=D, x=Vec(x), b=Vec(b), dinv=Vec(dinv), x1=Vec(torch.empty_like(x)), r=Vec(torch.empty_like(x)),
                 norm=Vec(torch.empty(1, dtype=torch.float64, device=DEV)))
    elif kind == "transfer":
        fine, coarse = _vectors(case, seed)
        s.update(fine=Vec(fine), coarse=Vec(coarse), down=Vec(torch.empty_like(coarse)),
                 up=Vec(torch.empty_like(fine)), mask=(ctypes.c_uint64 * 8)(*[2] * 8))
    elif kind == "cg":
        b = _vectors(case, seed)
        D, _ = _q1(case["side"], "f64")
        s.update(D=D, b=Vec(b), x=Vec(torch.empty_like(b)))
    elif kind == "pcg":
        coeff, b = _vectors(case, seed)
        D, dinv = _q1(case["side"], "f64", omega=1.0, coeff=coeff)
        _drop_boundary_columns(D, case["side"])
        s.update(D=D, b=Vec(b), dinv=Vec(dinv), x=Vec(torch.empty_like(b)))
    elif kind == "mixed":
        xt = _vectors(case, seed)
        D, _ = _q1(2 ** case["level"] + 1, "f64")
        b = Vec(torch.empty_like(xt))
        D.product(b, Vec(xt))
        torch.cuda.synchronize()
        mg = H.Multigrid(VT[case["inner"]], 1, case["level"])
        mg.configure(H.mg_config(n_max_iter=1, tolerance=1e-10, initial_zero=True, zero_inner_start=True))
        mg.build_q1(0.7)
        s.update(mg=mg, b=b, x=Vec(torch.empty_like(xt)))
    elif kind == "mgcg":
        coeff, b = _vectors(case, seed)
        torch.cuda.synchronize()
        mg = H.Multigrid(VT[case["inner"]], 1, case["level"])
        mg.configure(H.mg_config(n_max_iter=1, tolerance=1e-8))
        mg.build_q1_coeff(Vec(coeff), omega=0.8, averaging=1)
        s.update(mg=mg, coeff=coeff, b=Vec(b), x=Vec(torch.empty_like(b)))
    else:
        systems = _vectors(case, seed)
        levels = sorted({v for v, _, _ in systems}, reverse=True)
        counts = [sum(v == w for w, _, _ in systems) for v in levels]
        B = H.Batch(levels, counts, H.batch_config(inner_vtype=VT[case["inner"]], iters_per_launch=24,
                                                   first_launch_from_history=1))
        xs = [torch.empty(c, (2 ** v + 1) ** 2, dtype=torch.float64, device=DEV) for v, c in zip(levels, counts)]
        s.update(B=B, slots=[B.slot(i, j) for i, c in enumerate(counts) for j in range(c)],
                 coeffs=[Vec(c) for _, c, _ in systems], bs=[Vec(b) for _, _, b in systems], xs=xs,
                 rows=[Vec(x[j]) for x in xs for j in range(x.shape[0])])
    torch.cuda.synchronize()
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind in ("product", "random"):
        s["D"].product(s["y"], s["x"])
        return s["y"].t
    if kind == "sliced":
        s["S"].product(s["y"], s["x"])
        return s["y"].t
    if kind == "smooth":
        s["D"].jacobi(s["x1"], s["x"], s["b"], s["dinv"])
        if not case["host_norm"]:
            s["D"].defect_norm(s["r"], s["b"], s["x1"], s["norm"])
            return s["x1"].t, s["r"].t, s["norm"].t
        s["D"].defect(s["r"], s["b"], s["x1"])
        v, fn = ((ctypes.c_double(), "honei_hip_norm_l2_one_double") if case["dtype"] == "f64" else
                 (ctypes.c_float(), "honei_hip_norm_l2_one_float"))
        H.call(fn, ctypes.byref(v), s["r"].ptr, s["r"].n, None)
        return s["x1"].t, s["r"].t, np.array(v.value, np.float64 if case["dtype"] == "f64" else np.float32)
    if kind == "transfer":
        vt = VT[case["dtype"]]
        H.call("honei_hip_restriction", vt, s["down"].ptr, s["down"].n, s["fine"].ptr, s["fine"].n, s["mask"], None)
        H.call("honei_hip_prolongation", vt, s["up"].ptr, s["up"].n, s["coarse"].ptr, s["coarse"].n, s["mask"], None)
        return s["down"].t, s["up"].t
    if kind == "batch":
        B = s["B"]
        B.load_many(s["slots"], s["coeffs"], s["bs"])
        B.activate(True)
        B.run()
        for slot, x in zip(s["slots"], s["rows"]):
            B.result(slot, x)
        return s["xs"]
    x = s["x"]
    x.t.zero_()
    if kind == "cg":
        H.cg_solve(s["D"], s["b"], x, max_iters=10000, eps=1e-8)
    elif kind == "pcg":
        H.pcg_jacobi(s["D"], s["b"], x, s["dinv"], max_iters=20000, eps=1e-8)
    elif kind == "mixed":
        s["mg"].solve_mixed(s["b"], x)
    else:
        s["mg"].solve_pcg(s["b"], x)
    return x.t


# ---- what a pass cannot do without ---------------------------------------------
def work(case):
    """Operands read once and results written once.  A solve cannot do with
    less than its system and right-hand side in and the solution out; its
    operations are those of one cycle (multigrid) or of about 3 side
    iterations (Krylov methods) of the matrix alone."""
    kind = case["kind"]
    if kind in ("random", "sliced"):
        n, sv = case["n"], SIZE[case["dtype"]]
        nnz = n * (WIDTH + 1) // 2
        return {"bytes": nnz * (sv + 4) + 2 * n * sv, "flops": 2 * nnz}
    if kind in ("product", "smooth"):
        side, sv = case["side"], SIZE[case["dtype"]]
        n, nnz, sx = side * side, 9 * (side - 2) ** 2 + 4 * (side - 1), max(SIZE[case["dtype"]], 4)
        if kind == "product":
            return {"bytes": nnz * (sv + 4) + 2 * n * sx, "flops": 2 * nnz}
        return {"bytes": nnz * (sv + 4) + 5 * n * sx, "flops": 4 * nnz + 7 * n}
    if kind == "transfer":
        nf, nc, sv = (2 ** case["level"] + 1) ** 2, (2 ** (case["level"] - 1) + 1) ** 2, SIZE[case["dtype"]]
        return {"bytes": 2 * (nf + nc) * sv, "flops": 16 * nc + 4 * nf}
    if kind in ("cg", "pcg"):
        n = case["side"] ** 2
        return {"bytes": n * (9 * 12 + (24 if kind == "pcg" else 16)), "flops": 3 * case["side"] * 28 * n}
    if kind in ("mixed", "mgcg"):
        n = (2 ** case["level"] + 1) ** 2
        return {"bytes": n * (9 * 12 + 16), "flops": 9 * (4 * 22 * n * 4 // 3 + 20 * n)}
    n = sum(case["n%d" % v] * (2 ** v + 1) ** 2 for v in range(5, 10))
    return {"bytes": n * 24, "flops": 12 * (4 * 22 * n * 4 // 3 + 30 * n)}


# ---- the same in 64 bits ---------------------------------------------------------
def _edge(side):
    m = torch.zeros(side, side, dtype=torch.bool, device=DEV)
    m[0], m[-1], m[:, 0], m[:, -1] = True, True, True, True
    return m


def _stencil(x, off, mid):
    """Constant nine-point operator with identity boundary rows; x [side, side]."""
    y = x.clone()
    y[1:-1, 1:-1] *= mid - off
    inner = y[1:-1, 1:-1]
    side = x.shape[0]
    for i in range(3):
        for j in range(3):
            inner.add_(x[i:side - 2 + i, j:side - 2 + j], alpha=off)
    return y


def _poisson(coeff, b, coupled):
    """Solutions of a group of Q1 systems: coeff [k, c, c] per cell, b [k, s, s];
    conjugate gradients on the interior unknowns.  coupled: the interior rows
    keep their couplings to the boundary columns."""
    k, s = b.shape[0], b.shape[1]
    mask = (~_edge(s)).to(torch.float64)
    corner = -coeff / 3
    horiz = torch.zeros(k, s, s - 1, dtype=torch.float64, device=DEV)
    vert = torch.zeros(k, s - 1, s, dtype=torch.float64, device=DEV)
    diag = torch.zeros(k, s, s, dtype=torch.float64, device=DEV)
    for part in (horiz[:, :-1], horiz[:, 1:], vert[:, :, :-1], vert[:, :, 1:]):
        part -= coeff / 6
    for part in (diag[:, :-1, :-1], diag[:, :-1, 1:], diag[:, 1:, :-1], diag[:, 1:, 1:]):
        part += coeff * (2 / 3)

    def apply(p):
        y = diag * p
        y[:, :, :-1].addcmul_(horiz, p[:, :, 1:])
        y[:, :, 1:].addcmul_(horiz, p[:, :, :-1])
        y[:, :-1].addcmul_(vert, p[:, 1:])
        y[:, 1:].addcmul_(vert, p[:, :-1])
        y[:, :-1, :-1].addcmul_(corner, p[:, 1:, 1:])
        y[:, :-1, 1:].addcmul_(corner, p[:, 1:, :-1])
        y[:, 1:, :-1].addcmul_(corner, p[:, :-1, 1:])
        y[:, 1:, 1:].addcmul_(corner, p[:, :-1, :-1])
        return y.mul_(mask)

    dot = lambda u, v: (u * v).sum((1, 2), keepdim=True)
    x = b * (1 - mask)
    r = b * mask - (apply(x) if coupled else 0)
    z = r / diag
    p, rz, stop = z.clone(), dot(r, z), 1e-28 * dot(r, r)
    for it in range(40 * s):
        q = apply(p)
        a = rz / dot(p, q).clamp_min(1e-300)
        x.addcmul_(a, p)
        r.addcmul_(a, q, value=-1)
        z = r / diag
        new = dot(r, z)
        p.mul_(new / rz.clamp_min(1e-300)).add_(z)
        rz = new
        if it % 50 == 49 and bool((dot(r, r) <= stop).all()):
            break
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind in ("random", "sliced"):
        Aj, Ax, Arl, x = _random_arrays(case, seed)
        n, x = case["n"], x.double()
        y = torch.zeros(n, dtype=torch.float64, device=DEV)
        for k in range(WIDTH):
            y += torch.where(k < Arl, Ax[k, :n].double() * x[Aj[k, :n].long()], 0)
        return y
    if kind in ("product", "smooth"):
        side, dt = case["side"], VALUES[case["dtype"]]
        off, mid = (float(torch.tensor(v, dtype=torch.float64).to(TORCH[case["dtype"]]).to(dt)) for v in (-1 / 3, 8 / 3))
        x, b = (v.double().view(side, side) for v in _vectors(case, seed))
        if kind == "product":
            return _stencil(x, off, mid).view(-1)
        one = TORCH[case["dtype"]]
        w, d = torch.tensor(0.8, dtype=one), torch.tensor(mid, dtype=one)
        dinv = torch.full_like(x, float((1 / d) * w)).masked_fill_(_edge(side), float(w))
        x1 = x + dinv * (b - _stencil(x, off, mid))
        r = b - _stencil(x1, off, mid)
        if case["host_norm"]:
            return x1.view(-1), r.view(-1), np.array(float((r * r).sum()))
        return x1.view(-1), r.view(-1), (r * r).sum().view(1)
    if kind == "transfer":
        fine, coarse = (v.double() for v in _vectors(case, seed))
        sf, sc = 2 ** case["level"] + 1, 2 ** (case["level"] - 1) + 1
        f = torch.zeros(sf + 2, sf + 2, dtype=torch.float64, device=DEV)
        f[1:-1, 1:-1] = fine.view(sf, sf)
        down = torch.zeros(sc, sc, dtype=torch.float64, device=DEV)
        up = torch.zeros(sf + 2, sf + 2, dtype=torch.float64, device=DEV)
        for i in range(3):
            for j in range(3):
                w = 0.5 ** (abs(i - 1) + abs(j - 1))
                down += w * f[i:i + sf:2, j:j + sf:2]
                up[i:i + sf:2, j:j + sf:2] += w * coarse.view(sc, sc)
        return down.masked_fill(_edge(sc), 0).view(-1), up[1:-1, 1:-1].masked_fill(_edge(sf), 0).reshape(-1)
    if kind == "cg":
        side = case["side"]
        one = torch.ones(1, side - 1, side - 1, dtype=torch.float64, device=DEV)
        return _poisson(one, _vectors(case, seed).view(1, side, side), True).view(-1)
    if kind == "pcg":
        side, (coeff, b) = case["side"], _vectors(case, seed)
        return _poisson(coeff.view(1, side - 1, side - 1), b.view(1, side, side), False).view(-1)
    if kind == "mixed":
        return _vectors(case, seed)   # b is the product of these values
    if kind == "mgcg":
        side, (coeff, b) = 2 ** case["level"] + 1, _vectors(case, seed)
        return _poisson(coeff.view(1, side - 1, side - 1), b.view(1, side, side), True).view(-1)
    groups = {}
    for level, coeff, b in _vectors(case, seed):
        groups.setdefault(level, []).append((coeff, b))
    out = []
    for level, group in groups.items():
        side = 2 ** level + 1
        x = _poisson(torch.stack([c for c, _ in group]).view(-1, side - 1, side - 1),
                     torch.stack([b for _, b in group]).view(-1, side, side), True)
        out.append(x.view(len(group), -1))
    return out
