"""The workloads by which this framework's speed is followed.

Each case is one piece of work as a program using the framework asks for it: a whole solve
(PCG around a multigrid V-cycle, the Stokes multigrid, a batch of solves, PCG around an
incomplete factorisation), or one call that a solver loop of its own makes (a smoother call,
a sparse matrix-vector product, a training step of the learned smoother's network).

listed() names the cases, draw(rng) gives more of the same ranges, prepare() builds what the
program holds before the call, run() makes the call, exact() repeats it in plain 64-bit torch.
"""
import importlib.util
import itertools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _feat():
    """The package (its directory name has a dot, so it is imported by path)."""
    if "feat3amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location("feat3amd", os.path.join(
            os.getcwd() if os.path.isdir("feat3.doxytest_amd") else _ROOT, "feat3.doxytest_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules["feat3amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["feat3amd"]


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest whole solve in use (1,089 unknowns): launches and host latency count.
        # graphs: the solver replays recorded launches (its default) or issues them one by one;
        # nu: smoothing steps before and after the coarse correction
        dict(name="poisson2d_l5", kind="solve", dim=2, level=5, coef="constant", precision="f64", graphs=True, nu=4),
        # the framework's benchmark: 2.1 M unknowns, constant coefficient
        dict(name="poisson3d_l7", kind="solve", dim=3, level=7, coef="constant", precision="f64", graphs=False, nu=4),
        # an anisotropic log-normal medium, 275 k unknowns: matrices with all values distinct
        dict(name="diffusion3d_l6", kind="solve", dim=3, level=6, coef="lognormal", precision="f64", graphs=False, nu=4),
        # the same kind of problem with the mixed-precision cycle (FP16-valued matrices)
        dict(name="diffusion3d_l6_f16", kind="solve", dim=3, level=6, coef="lognormal", precision="f16", graphs=True, nu=4),
        # one smoother call (4 damped Jacobi steps and the last defect) of a variable-coefficient
        # fine level with 2.1 M unknowns, as a solver loop of one's own makes it
        dict(name="smooth3d_129", kind="smooth", dim=3, n1=129, precision="f64", steps=4),
        # r = y + a A x in the caller's CSR arrays on the benchmark's matrix (57 M entries)
        dict(name="spmv_q1_l7", kind="spmv_q1", dim=3, level=7, transposed=False),
        # the same product on an irregular matrix (0 to 40 entries a row), 32-bit values and indices
        dict(name="spmv_ragged_f32", kind="spmv", rows=300007, cols=290011, maxlen=40, values="f32", index="u32",
             transposed=False),
        # r = y + a A^T x without a stored transpose
        dict(name="spmv_transposed_l6", kind="spmv_q1", dim=3, level=6, transposed=True),
        # lid-driven cavity, Q2/P1dc, 45 k unknowns: Vanka-smoothed multigrid
        dict(name="stokes_l6", kind="stokes", level=6, steps=5),
        # 64 independent diffusion problems of uneven sizes (81 to 66,049 unknowns) at once;
        # mix picks the sizes and the media
        dict(name="batch_64", kind="batch", ninst=64, lmin=3, lmax=8, mix=1),
        # PCG around ILU(0): no hierarchy at hand
        dict(name="pcg_ilu_3d_l5", kind="krylov", dim=3, level=5, precond="ilu"),
        # the learned smoother's network: prediction, gradient and Adam step over a field's samples
        dict(name="learn_33", kind="learn", m=33),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "smooth", "smooth", "spmv", "spmv", "stokes", "batch", "krylov", "learn"])
    if kind == "solve":
        coef, precision = rng.choice(["constant", "lognormal"]), rng.choice(["f64", "f64", "f32", "f16"])
        dim, graphs = rng.choice([2, 3]), rng.random() < 0.5
        low, high = (3, 9 if coef == "constant" else 8) if dim == 2 else (2, 7 if coef == "constant" else 6)
        return dict(kind=kind, dim=dim, level=rng.randint(low, high), coef=coef, precision=precision, graphs=graphs,
                    nu=rng.choice([2, 3, 4, 4]))
    if kind == "smooth":
        dim = rng.choice([2, 3, 3])
        return dict(kind=kind, dim=dim, n1=_log_int(rng, 9, 1025) if dim == 2 else _log_int(rng, 5, 129),
                    precision=rng.choice(["f64", "f32", "f16"]), steps=rng.randint(1, 5))
    if kind == "spmv":
        rows = _log_int(rng, 500, 1000000)
        return dict(kind=kind, rows=rows, cols=max(1, int(rows * rng.uniform(0.3, 2.0))), maxlen=_log_int(rng, 6, 60),
                    values=rng.choice(["f64", "f32"]), index=rng.choice(["u64", "u32"]),
                    transposed=rng.random() < 0.35)
    if kind == "stokes":
        return dict(kind=kind, level=rng.randint(3, 6), steps=rng.choice([3, 4, 5]))
    if kind == "batch":
        lmin = rng.randint(2, 5)
        return dict(kind=kind, ninst=_log_int(rng, 3, 64), lmin=lmin, lmax=rng.randint(lmin + 1, 8),
                    mix=rng.randint(2, 1 << 20))
    if kind == "krylov":
        dim = rng.choice([2, 3])
        return dict(kind=kind, dim=dim, level=rng.randint(4, 6) if dim == 2 else rng.randint(3, 5),
                    precond=rng.choice(["ilu", "ssor", "jacobi"]))
    return dict(kind="learn", m=_log_int(rng, 9, 65))


# ---------------------------------------------------------------- inputs
_KZ, _SIGMA3, _SIGMA2 = 10.0, 1.5, 1.0   # anisotropy, and the spread of the log-normal coefficient
_OMEGA = 0.5                             # Jacobi damping of every smoother


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 2654435761 % (1 << 62))


def _uniform(g, n):
    """n values in [-1, 1] (right-hand sides)."""
    return torch.rand(n, generator=g, dtype=torch.float64, device="cuda") * 2 - 1


def _boundary(dim, n1):
    """True on the boundary nodes of an n1^dim grid."""
    m = torch.ones((n1,) * dim, dtype=torch.bool, device="cuda")
    m[(slice(1, -1),) * dim] = False
    return m


def _cells(case, seed):
    """The coefficient of every finest cell, or None where it is 1."""
    if case["coef"] == "constant":
        return None
    ncell = 1 << (case["dim"] * case["level"])
    z = torch.randn(ncell, generator=_gen(seed + 77), dtype=torch.float64, device="cuda")
    return torch.exp((_SIGMA3 if case["dim"] == 3 else _SIGMA2) * z)


def _load(case, seed):
    """Right-hand side, zero on the boundary."""
    n1 = (1 << case["level"]) + 1
    b = _uniform(_gen(seed), n1 ** case["dim"])
    b[_boundary(case["dim"], n1).reshape(-1)] = 0.0
    return b


def _slots(dim, n1, coef, h_power=0):
    """The clipped 3^dim-point matrix of -div(c K grad u), bilinear / trilinear elements, on an
    n1^dim grid: a list of 3^dim tensors in ascending column order, 0 outside the grid.  coef: one
    value for each cell and Gauss point, (2^dim,) + (n1-1,)*dim with the slowest axis first, or None."""
    off = list(itertools.product((-1, 0, 1), repeat=dim))
    val = [torch.zeros((n1,) * dim, dtype=torch.float64, device="cuda") for _ in off]
    g = 1 / math.sqrt(3.0)
    kdir = [_KZ if (dim == 3 and k == 0 and coef is not None) else 1.0 for k in range(dim)]   # axis 0 = z
    corners = list(itertools.product((0, 1), repeat=dim))
    gauss = list(itertools.product((-g, g), repeat=dim))
    grad = []
    for p in gauss:
        rows = []
        for a in corners:
            line = [(1 + p[k]) / 2 if a[k] else (1 - p[k]) / 2 for k in range(dim)]
            rows.append([math.prod((0.5 if a[j] else -0.5) if j == k else line[j] for j in range(dim)) for k in range(dim)])
        grad.append(rows)
    scale = (0.5 / (n1 - 1)) ** (dim - 2)
    for a, b in itertools.product(range(len(corners)), repeat=2):
        w = [sum(kdir[k] * grad[q][a][k] * grad[q][b][k] for k in range(dim)) for q in range(len(gauss))]
        at = tuple(slice(corners[a][k], n1 - 1 + corners[a][k]) for k in range(dim))
        t = off.index(tuple(corners[b][k] - corners[a][k] for k in range(dim)))
        if coef is None:
            val[t][at] += scale * math.fsum(w)
        else:
            val[t][at] += scale * sum(wq * coef[q] for q, wq in enumerate(w))
    return off, val


def _sampled(cells, dim, level, fine):
    """cells (finest level) at the Gauss points of every cell of `level`."""
    if cells is None:
        return None
    c = cells.reshape((1 << fine,) * dim)
    m, g = 1 << (fine - level), 1 / math.sqrt(3.0)
    at = [min(m - 1, int(m * (1 + s) / 2)) for s in (-g, g)]
    return torch.stack([c[tuple(slice(at[i], None, m) for i in q)] for q in itertools.product((0, 1), repeat=dim)])


def _csr_of_slots(dim, n1, off, val):
    """The slots inside the grid as CSR arrays (int64 indices)."""
    n = n1 ** dim
    node = torch.arange(n, device="cuda").reshape((n1,) * dim)
    inside, cols = [], []
    for o in off:
        ok = torch.ones((n1,) * dim, dtype=torch.bool, device="cuda")
        for k, d in enumerate(o):
            ix = torch.arange(n1, device="cuda") + d
            ok &= ((ix >= 0) & (ix < n1)).reshape([-1 if j == k else 1 for j in range(dim)])
        inside.append(ok.reshape(-1))
        cols.append(node.reshape(-1) + sum(d * n1 ** (dim - 1 - k) for k, d in enumerate(o)))
    ins = torch.stack(inside, 1)
    rowptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    rowptr[1:] = torch.cumsum(ins.sum(1), 0)
    return torch.stack([v.reshape(-1) for v in val], 1)[ins], torch.stack(cols, 1)[ins], rowptr


def _smooth_inputs(case, seed):
    """A random medium's matrix on an n1^dim grid, and the smoother's right-hand side."""
    dim, n1 = case["dim"], case["n1"]
    c = torch.exp(1.5 * torch.randn((n1 - 1,) * dim, generator=_gen(seed + 5), dtype=torch.float64, device="cuda"))
    off, val = _slots(dim, n1, c.expand((2 ** dim,) + c.shape))
    rhs = _uniform(_gen(seed), n1 ** dim).reshape((n1,) * dim)
    rhs[_boundary(dim, n1)] = 0.0
    return off, val, rhs


def _ragged(case, seed):
    """An irregular CSR matrix (rows of 0 to maxlen entries, columns spread around the diagonal)
    and the vectors of r = y + a A^(T) x."""
    g = _gen(seed)
    rows, cols = case["rows"], case["cols"]
    length = torch.randint(0, case["maxlen"] + 1, (rows,), generator=g, device="cuda")
    rowptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    rowptr[1:] = torch.cumsum(length, 0)
    nnz = int(rowptr[-1])
    row = torch.repeat_interleave(torch.arange(rows, device="cuda"), length, output_size=nnz)
    spread = torch.randn(nnz, generator=g, device="cuda") * max(8.0, cols / 200)
    col = (row.double() * (cols / rows) + spread).round().long().clamp_(0, cols - 1)
    order = torch.argsort(row * cols + col)
    col = col[order]
    dt = torch.float64 if case["values"] == "f64" else torch.float32
    val = (torch.randn(nnz, generator=g, dtype=torch.float64, device="cuda")).to(dt)
    nx, nr = (rows, cols) if case["transposed"] else (cols, rows)
    return val, col, rowptr, row, _uniform(g, nx).to(dt), _uniform(g, nr).to(dt)


_ALPHA, _BETA = 0.75, 1.0


def _learn_inputs(case, seed):
    """Samples of a field of m^3 nodes (54 inputs in [-1, 1], padded to 64), targets, and the
    network's parameters and Adam state in FP32 (a network that has been trained for a while)."""
    g = _gen(seed)
    n = case["m"] ** 3
    X = torch.zeros((n, 64), dtype=torch.bfloat16, device="cuda")
    X[:, :54] = (torch.rand((n, 54), generator=g, device="cuda") * 2 - 1).to(torch.bfloat16)
    t = torch.randn(n, generator=g, device="cuda") * 0.3
    p = torch.zeros(8385, device="cuda")
    p[0:4096] = torch.randn(4096, generator=g, device="cuda") / 7
    p[0:4096].view(64, 64)[:, 54:] = 0
    p[4096:4160] = torch.randn(64, generator=g, device="cuda") * 0.1
    p[4160:8256] = torch.randn(4096, generator=g, device="cuda") / 8
    p[8256:8320] = torch.randn(64, generator=g, device="cuda") * 0.1
    p[8320:8384] = torch.randn(64, generator=g, device="cuda") / 8
    m = torch.randn(8385, generator=g, device="cuda") * 1e-2
    m[0:4096].view(64, 64)[:, 54:] = 0
    v = torch.rand(8385, generator=g, device="cuda") * 1e-3 + 1e-4
    return X, t, p, m, v


_ADAM = dict(step=100, lr=1e-3, b1=0.9, b2=0.999, eps=1e-8)


# ---------------------------------------------------------------- prepare / run
def _levels(F, case, seed):
    """Host levels of a log-normal hierarchy, finest first."""
    dim, fine = case["dim"], case["level"]
    cells = _cells(case, seed).cpu().numpy()
    out = []
    for k in range(fine, 0, -1):
        q = dict(F.q1_problem(dim, k))
        q["val"] = F.q1_diffusion3d(k, fine, cells, _KZ) if dim == 3 else F.q1_diffusion(k, fine, cells)
        out.append(q)
    return out


def prepare(case, seed):
    F = _feat()
    F.libs()
    kind = case["kind"]
    if kind == "solve":
        cfg = F.mgpcg_cfg(nu_pre=case["nu"], nu_post=case["nu"], omega_jac=_OMEGA, coarse="direct", tol_rel=1e-8, max_iter=200,
                          precision=case["precision"], graphs=case["graphs"])
        if case["coef"] == "constant":
            s = F.MgPcg(cfg, q1=(case["dim"], case["level"], 1))
        else:
            s = F.MgPcg(cfg, levels=_levels(F, case, seed))
        b = _load(case, seed)
        return dict(kind=kind, solver=s, x=torch.zeros_like(b), b=b)
    if kind == "krylov":
        q = F.q1_problem(case["dim"], case["level"])

        class A:
            rows, val, col, rowptr = q["n"], q["val"], q["col"], q["rowptr"]
        omega = 0.0 if case["precond"] == "ilu" else 1.0   # ILU: the fill level
        s = F.KrylovSolver("pcg", A, q["filt"], case["precond"], omega_pre=omega, tol_rel=1e-8, max_iter=2000)
        b = _load(case, seed)
        return dict(kind="solve", solver=s, x=torch.zeros_like(b), b=b)
    if kind == "stokes":
        s = F.Stokes(case["level"], 1, steps=case["steps"], omega_rich=0.7, tol_rel=1e-8, max_iter=100)
        nv, n = s.sizes(0)["nv"], s.n(0)
        b = torch.zeros(n, dtype=torch.float64, device="cuda")
        b[:2 * nv] = _uniform(_gen(seed), 2 * nv) / nv   # a rough body force; the lid moves as well
        x0 = torch.zeros(n, dtype=torch.float64, device="cuda")
        s.filter(0, b, "rhs")
        s.filter(0, x0, "sol")
        return dict(kind=kind, solver=s, x=torch.empty_like(x0), x0=x0, b=b)
    if kind == "batch":
        s = F.BatchSolver(seed=case["mix"], ninst=case["ninst"], lmin=case["lmin"], lmax=case["lmax"], sigma=_SIGMA2,
                          tol_rel=1e-8, max_iter=100)
        b = torch.from_numpy(F.batch_rhs(s, int(seed) + 1)).cuda()
        return dict(kind="solve", solver=s, x=torch.zeros_like(b), b=b)
    h = F.Handle(0, stream=torch.cuda.current_stream().cuda_stream)
    if kind == "smooth":
        off, val, rhs = _smooth_inputs(case, seed)
        dim, n1, fp = case["dim"], case["n1"], case["precision"]
        n = n1 ** dim
        diag = val[len(off) // 2].reshape(-1)
        plan = F.SellPlan(h, *_csr_of_slots(dim, n1, off, val), n, n, fp=fp)
        dt = torch.float64 if fp == "f64" else torch.float32
        idx = torch.nonzero(_boundary(dim, n1).reshape(-1)).reshape(-1)
        mask = torch.zeros((n + 31) // 32, dtype=torch.int32, device="cuda")
        F.check(h.k.feat_unit_filter_mask_u64(h.h, F.ptr(mask), n, F.ptr(idx), idx.numel()), "mask")
        keep, ws = F.reduce_ws(torch, "cuda")
        new = lambda: torch.empty(n, dtype=dt, device="cuda")
        return dict(kind=kind, h=h, plan=plan, fp=fp, steps=case["steps"], inv=(_OMEGA / diag).to(dt), mask=mask,
                    rhs=rhs.reshape(-1).to(dt), x=new(), tmp=new(), d=new(), keep=(keep, idx), ws=ws)
    if kind == "spmv_q1":
        q = F.q1_problem_device(torch, h, case["dim"], case["level"], transfer=False)
        g = _gen(seed)
        val = q["val"] * (1 + 0.1 * _uniform(g, q["val"].numel()))   # values of its own in every entry
        return dict(kind="spmv", h=h, fn=h.k.feat_csr_apply_f64_u64, val=val, col=q["col"], rowptr=q["rowptr"],
                    rows=q["n"], cols=q["n"], x=_uniform(g, q["n"]), y=_uniform(g, q["n"]),
                    r=torch.empty(q["n"], dtype=torch.float64, device="cuda"), t=int(case["transposed"]))
    if kind == "spmv":
        val, col, rowptr, _, x, y = _ragged(case, seed)
        if case["index"] == "u32":
            col, rowptr = col.int(), rowptr.int()
        fn = getattr(h.k, "feat_csr_apply_%s_%s" % (case["values"], case["index"]))
        return dict(kind=kind, h=h, fn=fn, val=val, col=col, rowptr=rowptr, rows=case["rows"], cols=case["cols"], x=x,
                    y=y, r=torch.empty_like(y), t=int(case["transposed"]))
    X, t, p, m, v = _learn_inputs(case, seed)
    n = t.numel()
    wbf = torch.empty(8192, dtype=torch.bfloat16, device="cuda")
    F.check(h.k.feat_mlp_to_bf16(h.h, F.ptr(p), F.ptr(wbf)), "feat_mlp_to_bf16")
    return dict(kind="learn", h=h, X=X, t=t, p=p, m=m, v=v, wbf=wbf, n=n, step=_ADAM["step"],
                y=torch.empty(n, device="cuda"), grad=torch.empty(8448, device="cuda"),
                part=torch.empty(1056 * 8448, device="cuda"))


def run(state):
    F = _feat()
    kind = state["kind"]
    if kind == "solve":
        state["x"].zero_()
        state["solver"].solve(state["x"], state["b"])
        return {"x": state["x"]}
    if kind == "stokes":
        state["x"].copy_(state["x0"])
        state["solver"].solve(state["x"], state["b"])
        return {"x": state["x"]}
    h, P = state["h"], F.ptr
    if kind == "smooth":
        a = (h.h, state["plan"].m, P(state["inv"]), P(state["mask"]), state["steps"], _OMEGA_RICH, P(state["rhs"]), None,
             P(state["x"]), P(state["tmp"]), P(state["d"]), None)
        if state["fp"] == "f64":
            F.check(h.k.feat_rj_smooth_f64(*a, None, None, state["ws"]), "feat_rj_smooth_f64")
        else:
            F.check(h.k.feat_rj_smooth_f32(*a, state["ws"]), "feat_rj_smooth_f32")
        return {"x": state["x"], "defect": state["d"]}
    if kind == "spmv":
        F.check(state["fn"](h.h, P(state["r"]), _ALPHA, P(state["x"]), _BETA, P(state["y"]), P(state["val"]),
                            P(state["col"]), P(state["rowptr"]), state["rows"], state["cols"], state["val"].numel(),
                            state["t"]), "feat_csr_apply")
        return {"r": state["r"]}
    n, k = state["n"], h.k
    F.check(k.feat_mlp_infer(h.h, P(state["p"]), P(state["wbf"]), P(state["X"]), n, P(state["y"])), "feat_mlp_infer")
    F.check(k.feat_mlp_grad(h.h, P(state["p"]), P(state["wbf"]), P(state["X"]), P(state["t"]), n, P(state["part"]), 1056,
                            P(state["grad"])), "feat_mlp_grad")
    F.check(k.feat_mlp_adam(h.h, P(state["p"]), P(state["wbf"]), P(state["grad"]), P(state["m"]), P(state["v"]),
                            state["step"], _ADAM["lr"], _ADAM["b1"], _ADAM["b2"], _ADAM["eps"]), "feat_mlp_adam")
    state["step"] += 1
    return {"y": state["y"], "grad": state["grad"][:8385], "p": state["p"], "m": state["m"], "v": state["v"]}


_OMEGA_RICH = 1.0   # Richardson damping of the smoothers


# ---------------------------------------------------------------- work and tolerance
def _stencil_nnz(dim, n1):
    return (3 * n1 - 2) ** dim


def work(case):
    """Bytes of the inputs and outputs, and the operations of the method (for the solves: of the
    usual number of iterations, 2 nu + 3 finest-level products each, and the coarser levels)."""
    kind = case["kind"]
    if kind in ("solve", "krylov"):
        dim, n1 = case["dim"], (1 << case["level"]) + 1
        n, nnz = n1 ** dim, _stencil_nnz(case["dim"], n1)
        if kind == "krylov":
            return {"bytes": 8 * nnz + 16 * n, "flops": 30 * (4 * nnz + 10 * n)}
        vbytes = 0 if case["coef"] == "constant" else 8 * nnz
        its = 5 if case["coef"] == "constant" else 40 if dim == 3 else 12
        return {"bytes": vbytes + 16 * n, "flops": its * ((4 * case["nu"] + 6) * nnz + 40 * n) * (8 / 7 if dim == 3 else 4 / 3)}
    if kind == "stokes":
        cells = 4 ** case["level"]
        nnz = 4 * 16 * 4 * cells + 4 * 54 * cells   # velocity entries and the two couplings
        return {"bytes": 8 * nnz + 16 * 11 * cells, "flops": 10 * (2 * case["steps"] + 2) * 6 * nnz * 4 / 3}
    if kind == "batch":
        per = [((1 << lv) + 1) ** 2 for lv in range(case["lmin"], case["lmax"] + 1)]
        n = case["ninst"] * sum(per) / len(per)
        return {"bytes": 9 * 8 * n + 16 * n, "flops": 12 * n * (22 * 9 + 40) * 4 / 3}
    if kind == "smooth":
        n, nnz = case["n1"] ** case["dim"], _stencil_nnz(case["dim"], case["n1"])
        size = {"f64": 8, "f32": 4, "f16": 2}[case["precision"]]
        vec = 8 if case["precision"] == "f64" else 4
        return {"bytes": size * nnz + 4 * vec * n + n / 8, "flops": case["steps"] * (2 * nnz + 4 * n)}
    if kind == "spmv_q1":
        n1 = (1 << case["level"]) + 1
        rows = cols = n1 ** case["dim"]
        nnz, size, index = _stencil_nnz(case["dim"], n1), 8, 8
    elif kind == "spmv":
        rows, cols, nnz = case["rows"], case["cols"], case["rows"] * case["maxlen"] / 2
        size, index = 8 if case["values"] == "f64" else 4, 8 if case["index"] == "u64" else 4
    else:
        n = case["m"] ** 3
        return {"bytes": n * (128 + 8) + 8385 * 4 * 7, "flops": 2.0 * n * (2 * 54 * 64 + 64 * 64 * 4 + 64 * 54)}
    nx, nr = (rows, cols) if case["transposed"] else (cols, rows)
    return {"bytes": nnz * (size + index) + (rows + 1) * index + size * (nx + 2 * nr), "flops": 2.0 * nnz}


def tolerance(case):
    """About four times what another order of the sums was seen to change."""
    kind = case["kind"]
    if kind == "solve":
        # a constant coefficient: 8e-14 from the 64-bit restatement.  The random media are badly
        # conditioned: the defects' history moves by some per cent with the last bits of the
        # right-hand side, so the step at which 1e-8 is reached can change
        if case["precision"] == "f64" and case["coef"] == "constant":
            return {"rel": 1e-12, "max": 1e-10}
        return {"rel": 2e-8, "max": 1e-6}
    if kind in ("stokes", "batch", "krylov"):
        return {"rel": 1e-9, "max": 1e-7}
    if kind == "learn":   # BF16 activations
        return {"rel": 7e-3, "max": 0.3}
    if kind == "smooth":
        return {"rel": 4e-15, "max": 1e-12} if case["precision"] == "f64" else {"rel": 1e-6, "max": 1e-4}
    return {"rel": 1e-15, "max": 1e-12} if case.get("values", "f64") == "f64" else {"rel": 5e-7, "max": 2e-5}


# ---------------------------------------------------------------- the same in plain 64-bit torch
class _Grid:
    """One multigrid level: the clipped stencil, the Dirichlet boundary, damped Jacobi."""

    def __init__(self, dim, level, fine, cells):
        self.dim, self.n1 = dim, (1 << level) + 1
        self.off, self.val = _slots(dim, self.n1, _sampled(cells, dim, level, fine))
        self.inside = (~_boundary(dim, self.n1)).double()
        self.inv = _OMEGA / self.val[len(self.off) // 2]

    def apply(self, x):
        p = torch.nn.functional.pad(x, (1, 1) * self.dim)
        r = torch.zeros_like(x)
        for o, v in zip(self.off, self.val):
            r += v * p[tuple(slice(1 + d, 1 + d + self.n1) for d in o)]
        return r

    def defect(self, b, x):
        return (b - self.apply(x)) * self.inside

    def smooth(self, b, steps, x=None):
        x = torch.zeros_like(b)
        d = b * self.inside
        for k in range(steps):
            x = x + self.inv * d * self.inside
            d = self.defect(b, x)
        return x, d

    def prolongate(self, c):
        f = torch.zeros((self.n1,) * self.dim, dtype=torch.float64, device="cuda")
        for q in itertools.product((0, 1), repeat=self.dim):      # the parity of the fine node
            s = 0
            for e in itertools.product(*[(0, 1) if i else (0,) for i in q]):
                s = s + c[tuple(slice(e[k], c.shape[k] - (q[k] - e[k])) for k in range(self.dim))]
            f[tuple(slice(i, None, 2) for i in q)] = s / 2 ** sum(q)
        return f

    def restrict(self, d):
        p = torch.nn.functional.pad(d, (1, 1) * self.dim)
        r = 0
        for o in self.off:
            w = 0.5 ** sum(abs(i) for i in o)
            r = r + w * p[tuple(slice(1 + i, 1 + i + self.n1, 2) for i in o)]
        return r


def _cycle(grids, i, b, nu):
    g = grids[i]
    if i + 1 == len(grids):   # one free node on level 1
        mid = (1,) * g.dim
        x = torch.zeros_like(b)
        x[mid] = b[mid] / g.val[len(g.off) // 2][mid]
        return x
    x, d = g.smooth(b, nu)
    c = _cycle(grids, i + 1, g.restrict(d) * grids[i + 1].inside, nu)
    x = x + g.prolongate(c) * g.inside
    return x + g.smooth(g.defect(b, x), nu)[0]


def _pcg(dim, level, cells, b, nu=4, tol=1e-8, most=200):
    grids = [_Grid(dim, k, level, cells) for k in range(level, 0, -1)]
    g = grids[0]
    b = b.reshape((g.n1,) * dim)
    x, r = torch.zeros_like(b), b * g.inside
    first = float(torch.linalg.vector_norm(r))
    z = _cycle(grids, 0, r, nu)
    p, gamma = z, (z * r).sum()
    for _ in range(most):
        q = g.apply(p) * g.inside
        alpha = gamma / (q * p).sum()
        x = x + alpha * p
        r = r - alpha * q
        if float(torch.linalg.vector_norm(r)) <= tol * first:
            break
        z = _cycle(grids, 0, r, nu)
        new = (z * r).sum()
        p, gamma = z + (new / gamma) * p, new
    return x.reshape(-1)


def _exact_learn(case, seed):
    X, t, p, m, v = (a.double() for a in _learn_inputs(case, seed))
    w = p.to(torch.bfloat16).double()   # the products take BF16 weights
    W1, b1, W2 = w[0:4096].view(64, 64), p[4096:4160], w[4160:8256].view(64, 64)
    b2, w3, b3 = p[8256:8320], p[8320:8384], p[8384]
    act = lambda z: 0.5 * z * (1 + torch.erf(z / math.sqrt(2.0)))
    slope = lambda z: 0.5 * (1 + torch.erf(z / math.sqrt(2.0))) + z * torch.exp(-z * z / 2) / math.sqrt(2 * math.pi)
    z1 = X @ W1.T + b1
    h1 = act(z1)
    z2 = h1 @ W2.T + b2
    h2 = act(z2)
    y = h2 @ w3 + b3
    e = 2 * (y - t) / t.numel()
    d2 = e[:, None] * w3 * slope(z2)
    d1 = (d2 @ W2) * slope(z1)
    g = torch.cat([(d1.T @ X).reshape(-1), d1.sum(0), (d2.T @ h1).reshape(-1), d2.sum(0), h2.T @ e, e.sum()[None]])
    m = _ADAM["b1"] * m + (1 - _ADAM["b1"]) * g
    v = _ADAM["b2"] * v + (1 - _ADAM["b2"]) * g * g
    k = _ADAM["step"]
    p = p - _ADAM["lr"] * (m / (1 - _ADAM["b1"] ** k)) / ((v / (1 - _ADAM["b2"] ** k)).sqrt() + _ADAM["eps"])
    return {"y": y, "grad": g, "p": p, "m": m, "v": v}


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve":
        return {"x": _pcg(case["dim"], case["level"], _cells(case, seed), _load(case, seed), case["nu"])}
    if kind == "krylov":   # the solution itself (the solve stops at 1e-8)
        return {"x": _pcg(case["dim"], case["level"], None, _load(case, seed), tol=1e-12)}
    if kind == "batch":
        F = _feat()   # the instances' sizes, coefficients and right-hand sides are inputs
        levels = F.batch_levels(case["mix"], case["ninst"], case["lmin"], case["lmax"])

        class B:
            pass
        B.levels = levels
        B.off = np.concatenate([[0], np.cumsum([((1 << int(lv)) + 1) ** 2 for lv in levels])])
        b = torch.from_numpy(F.batch_rhs(B, int(seed) + 1)).cuda()
        out = []
        for i, lv in enumerate(int(v) for v in levels):
            cells = torch.from_numpy(F.lognormal_cells(case["mix"] + 1000 + i, 1 << (2 * lv), _SIGMA2)).cuda()
            out.append(_pcg(2, lv, cells, b[int(B.off[i]):int(B.off[i + 1])]))
        return {"x": torch.cat(out)}
    if kind == "smooth":
        off, val, rhs = _smooth_inputs(case, seed)
        dim = case["dim"]
        g = _Grid.__new__(_Grid)
        g.dim, g.n1, g.off, g.val = dim, case["n1"], off, val
        g.inside, g.inv = (~_boundary(dim, g.n1)).double(), _OMEGA / val[len(off) // 2]
        x, d = g.smooth(rhs, case["steps"])
        return {"x": x.reshape(-1), "defect": d.reshape(-1)}
    if kind in ("spmv", "spmv_q1"):
        if kind == "spmv":
            val, col, _, row, x, y = _ragged(case, seed)
        else:
            # the pattern of the grid; the values as prepare() scales them
            dim, n1 = case["dim"], (1 << case["level"]) + 1
            off, slots = _slots(dim, n1, None)
            val, col, rowptr = _csr_of_slots(dim, n1, off, slots)
            g = _gen(seed)
            val = val * (1 + 0.1 * _uniform(g, val.numel()))
            row = torch.repeat_interleave(torch.arange(n1 ** dim, device="cuda"), rowptr[1:] - rowptr[:-1])
            x, y = _uniform(g, n1 ** dim), _uniform(g, n1 ** dim)
        src, dst = (row, col) if case["transposed"] else (col, row)
        r = y.double() * _BETA
        return {"r": r.index_add_(0, dst, _ALPHA * val.double() * x.double()[src])}
    if kind == "learn":
        return _exact_learn(case, seed)
    return None   # Stokes: a dense factorisation of its 45 k unknowns would take minutes
