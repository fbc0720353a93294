"""What the performance of this framework is measured on.

Every case is one call that a program makes once its system is set up: a
V-cycle (the preconditioner), a whole FGMRES solve, a V-cycle or solves on
several right-hand sides, the raw fixed-point SpMV, a gradient of the learned
network.  The systems are the generated families of bench.py and the tests.
A program sets a system up once and then solves many right-hand sides with it,
so the hierarchy on the GPU is kept per system (`_plan`) and `prepare` makes
the right-hand side, the solver handle and the buffers.
"""
import ctypes
import functools
import math
import os
import sys
import types

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "sc23-ad_amd"))
import sc23ad as S  # noqa: E402

FRAC_BITS = 29  # what the driver's rule gives on these systems
RTOL = 1e-8
SMOOTHERS = {"sor": S.SOR, "block_sor": S.BLOCK_SOR, "jacobi_sor": S.JACOBI_SOR}
PRECISIONS = {"int": S.INT, "fp64": S.FP64, "fp32": S.FP32}
TORCH = {"int": torch.int32, "fp64": torch.float64, "fp32": torch.float32}
MLP_IN, MLP_H, MLP_OUT = 8, 32, 2


def _case(op, family="", side=0, precision="int", smoother="block_sor", nrhs=1, count=0):
    return {"op": op, "family": family, "side": side, "precision": precision,
            "smoother": smoother, "nrhs": nrhs, "count": count}


def listed():
    def named(name, *a, **k):
        return dict(_case(*a, **k), name=name)
    return [
        # the smallest call: one V-cycle of a small 2D system inside a caller's own Krylov loop
        named("vcycle_int_poisson2d_48_sor", "vcycle", "poisson2d", 48, smoother="sor"),
        # the preconditioner of the headline system
        named("vcycle_int_laplace3d_128", "vcycle", "laplace3d", 128),
        # the sequential smoother (the binding's default) in 3D: one dependency chain, wide levels
        named("vcycle_int_laplace3d_63_sor", "vcycle", "laplace3d", 63, smoother="sor"),
        # the CPU-sized solve of the reference's seq.exe
        named("solve_int_poisson2d_256_sor", "solve", "poisson2d", 256, smoother="sor"),
        # the headline: 3D Laplacian to 1e-8
        named("solve_int_laplace3d_128", "solve", "laplace3d", 128),
        # 27-point variable-coefficient anisotropic diffusion
        named("solve_int_diffusion27_64", "solve", "diffusion27", 64),
        # the floating-point solvers of the same call surface
        named("solve_fp64_laplace3d_96", "solve", "laplace3d", 96, precision="fp64"),
        named("solve_fp32_diffusion27_48", "solve", "diffusion27", 48, precision="fp32"),
        # several right-hand sides: a full block and a ragged small one
        named("block_vcycle_inclusions3d_96_x16", "block_vcycle", "inclusions3d", 96, nrhs=16),
        # uneven systems, four right-hand sides each, all at once
        named("batch_convdiff2d_16x4", "batch", "convdiff2d", nrhs=4, count=16),
        # the fixed-point SpMV on a caller's own CSR arrays
        named("spmv_int_diffusion27_95", "spmv_int", "diffusion27", 95),
        # one gradient of the learned per-level network over a whole sweep's levels
        named("mlp_grad_1220", "mlp_grad", count=1220),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# largest sides drawn: 3D systems by what a pass on them costs
_SIDES = {"poisson2d": (24, 256), "convdiff2d": (32, 256), "laplace3d": (10, 128),
          "diffusion27": (10, 64), "inclusions3d": (12, 96)}


def draw(rng):
    op = rng.choice(["vcycle", "vcycle", "vcycle", "solve", "solve", "solve", "block_vcycle",
                     "block_vcycle", "batch", "spmv_int", "mlp_grad"])
    if op == "mlp_grad":
        return _case(op, count=_log(rng, 1, 4000))
    if op == "batch":
        return _case(op, "convdiff2d", nrhs=rng.randint(1, 6), count=rng.randint(2, 16))
    family = rng.choice(sorted(_SIDES))
    lo, hi = _SIDES[family]
    if op == "spmv_int":
        return _case(op, family, _log(rng, lo, hi))
    if op == "block_vcycle":
        return _case(op, family, _log(rng, lo, min(hi, 256 if "2d" in family else 96)),
                     nrhs=rng.randint(2, 16))
    precision = rng.choice(["int", "int", "fp64", "fp32"])
    if op == "solve" and family == "inclusions3d":  # the integer solver needs hundreds of steps
        precision = rng.choice(["fp64", "fp32"])
    if precision != "int":
        hi = min(hi, 256 if "2d" in family else 80)
    smoother = "block_sor"
    if "2d" in family:
        smoother = rng.choice(["sor", "block_sor"])
    elif op == "vcycle" and precision == "int":
        smoother = rng.choice(["sor", "block_sor", "block_sor", "jacobi_sor"])
        if smoother != "block_sor":
            hi = min(hi, 64)
    return _case(op, family, _log(rng, lo, hi), precision, smoother)


def _generate(family, side):
    """(kind, parameters) of a family at this side, as bench.py draws them."""
    if family == "poisson2d":
        return S.GEN_POISSON2D, (side,)
    if family == "laplace3d":
        return S.GEN_LAPLACE3D, (side,)
    if family == "diffusion27":
        return S.GEN_DIFFUSION27, (side, 8, 1.0, 1.0, 1e-3, 2)
    if family == "inclusions3d":  # spheres per volume of the 160^3 system with 64
        return S.GEN_INCLUSIONS3D, (side, max(1, round(64 * (side / 160) ** 3)), min(4, side / 6),
                                    min(12, side / 4), 1e6, 4)
    return S.GEN_CONVDIFF2D, (side, 40.0, 1.1)


def _setup(kind, params, precision, smoother):
    a = S.CsrMat.generate(kind, *params)
    a.lmax1_scaling(np.zeros(a.n))
    h = S.Hierarchy(a, PRECISIONS[precision], S.amg_param(SMOOTHERS[smoother]))
    return a, S.Amg(h)


@functools.lru_cache(maxsize=24)
def _plan(family, side, precision, smoother):
    """The row-scaled system and its hierarchy on the GPU."""
    return _setup(*_generate(family, side), precision, smoother)


@functools.lru_cache(maxsize=2)
def _batch_plan(count):
    n, pe, ang = S.convdiff_draws(256, 3)
    return [_setup(S.GEN_CONVDIFF2D, (int(n[k]), float(pe[k]), float(ang[k])), "int", "block_sor")
            for k in range(count)]


@functools.lru_cache(maxsize=4)
def _fixed_csr(family, side):
    """The system as 30-fractional-bit CSR arrays."""
    a = S.CsrMat.generate(*((k := _generate(family, side))[:1]), *k[1])
    a.lmax1_scaling(np.zeros(a.n))
    rptr, cind, val = a.arrays()
    return rptr, cind, np.trunc(val * 2.0 ** 30).astype(np.int32)


def _plan_of(case):
    return _plan(case["family"], case["side"], case["precision"], case["smoother"])


def _xstar(n, seed, k=0):
    return np.random.default_rng([seed, k]).uniform(-1.0, 1.0, n)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _dev(t):
    """A torch tensor as the device array the solvers take."""
    return types.SimpleNamespace(p=_ptr(t), nbytes=t.numel() * t.element_size())


def _krylov_like(shape, n, precision, seed):
    """A unit vector as the Krylov loop hands to the preconditioner (2^F fixed
    point for the integer solver)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.randn(shape, generator=g, device="cuda", dtype=torch.float64) / math.sqrt(n)
    return (v * 2.0 ** FRAC_BITS).to(torch.int32) if precision == "int" else v.to(TORCH[precision])


def _mlp_data(case, seed):
    """(W1, b1, W2, b2, W3, b3), features and targets."""
    r = np.random.default_rng(seed)
    w = []
    for out, inp in ((MLP_H, MLP_IN), (MLP_H, MLP_H), (MLP_OUT, MLP_H)):
        lim = math.sqrt(6.0 / (out + inp))
        w += [r.uniform(-lim, lim, (out, inp)).astype(np.float32),
              r.uniform(-0.1, 0.1, out).astype(np.float32)]
    return (w, r.uniform(0.0, 1.5, (case["count"], MLP_IN)).astype(np.float32),
            r.uniform(0.0, 1.0, (case["count"], MLP_OUT)).astype(np.float32))


def prepare(case, seed):
    op = case["op"]
    st = types.SimpleNamespace(op=op)
    if op == "mlp_grad":
        w, st.x, st.t = _mlp_data(case, seed)
        st.mlp = S.Mlp(0)
        st.mlp.set_params(np.concatenate([v.reshape(-1) for v in w]))
        return st
    if op == "batch":
        st.solvers, st.bs, st.nrm = [], [], []
        for k, (a, amg) in enumerate(_batch_plan(case["count"])):
            bs = [a.matvec(_xstar(a.n, seed, 64 * k + r)) for r in range(case["nrhs"])]
            st.bs.append(bs)
            st.nrm.append([float(np.linalg.norm(b)) for b in bs])
            st.solvers.append(S.BlockSolver(a, amg, [FRAC_BITS] * case["nrhs"], m=20, eps=RTOL,
                                            max_restarts=10))
        return st
    if op == "spmv_int":
        st.csr = [torch.from_numpy(v).cuda() for v in _fixed_csr(case["family"], case["side"])]
        n = len(st.csr[0]) - 1
        st.x = _krylov_like(n, n, "int", seed)
        st.y = torch.empty_like(st.x)
        torch.cuda.synchronize()
        return st
    a, st.amg = _plan_of(case)
    n = st.n = a.n
    if op == "vcycle":
        st.x = _krylov_like(n, n, case["precision"], seed)
        st.y = torch.empty_like(st.x)
    elif op == "block_vcycle":  # block layout: groups of four right-hand sides
        st.nrhs = case["nrhs"]
        st.x = _krylov_like(((st.nrhs + 3) // 4, n, 4), n, "int", seed)
        st.y = torch.empty_like(st.x)
    else:
        b = a.matvec(_xstar(n, seed))
        st.b = torch.from_numpy(b).cuda()
        st.nrm_b = float(np.linalg.norm(b))
        st.x = torch.empty_like(st.b)
        st.solver = S.Solver(PRECISIONS[case["precision"]], a, st.amg, eps=RTOL, bit=FRAC_BITS,
                             m=20 if case["family"] == "convdiff2d" else 30, max_restarts=5)
    torch.cuda.synchronize()
    return st


def run(st):
    if st.op == "mlp_grad":
        loss, grad = st.mlp.grad(st.x, st.t)
        return {"loss": loss, "grad": grad}
    if st.op == "batch":
        xs, cvs = S.block_solve_batch(st.solvers, st.bs, st.nrm)
        return {"x": np.concatenate([x.reshape(-1) for x in xs]),
                "iterations": np.array([c.iter for cv in cvs for c in cv]),
                "status": np.array([c.status for cv in cvs for c in cv])}
    if st.op == "spmv_int":
        rptr, cind, val = st.csr
        S.check(S.lib.sc23ad_spmv_int(len(rptr) - 1, _ptr(rptr), _ptr(cind), _ptr(val), 30,
                                      _ptr(st.x), _ptr(st.y)))
        return st.y
    if st.op == "vcycle":
        S.check(S.lib.sc23ad_amg_precondition(st.amg.h, _ptr(st.x), _ptr(st.y), 1))
        return st.y
    if st.op == "block_vcycle":
        S.check(S.lib.sc23ad_amg_precondition_block(st.amg.h, st.nrhs, _ptr(st.x), _ptr(st.y), 1))
        return st.y
    st.x.zero_()  # the initial guess
    torch.cuda.current_stream().synchronize()  # the solver works on a stream of its own
    cv = st.solver.solve_device(_dev(st.b), st.nrm_b, _dev(st.x))
    return {"x": st.x, "iterations": cv.iter, "status": cv.status}


def _vcycle_work(amg, nrhs=1):
    """Matrices read once, each right-hand side's vectors once per kernel."""
    es = np.dtype(amg.dtype).itemsize
    n = [float(v) for v in amg.level_n]
    vectors = sum(es * (13 * n[k] + 2 * n[k + 1]) for k in range(amg.depth)) + 4 * es * n[-1]
    matrices = max(0.0, amg.vcycle_bytes() - vectors)
    return {"bytes": matrices + nrhs * vectors, "flops": 2 * nrhs * matrices / (es + 4)}


def _solve_work(a, amg, m, nrhs=1):
    """One restart cycle of m steps: m V-cycles and products, the
    Gram-Schmidt passes, the outer residual and update."""
    es = np.dtype(amg.dtype).itemsize
    v = _vcycle_work(amg, nrhs)
    n, nnz = a.n, a.nnz
    spmv = (es + 4) * nnz + 4 * n + 2 * es * n * nrhs
    gs = es * n * (2.5 * m + 5) * nrhs
    return {"bytes": m * (v["bytes"] + spmv + gs) + 12 * nnz + (8 * 4 + es * m) * n * nrhs,
            "flops": m * (v["flops"] + 2 * nnz * nrhs + 2 * n * (m + 3) * nrhs) + 2 * nnz * nrhs}


def work(case):
    op = case["op"]
    if op == "mlp_grad":
        p = MLP_H * (MLP_IN + MLP_H + MLP_OUT)
        return {"bytes": 4 * case["count"] * (MLP_IN + MLP_OUT) + 8 * p,
                "flops": 6 * p * case["count"]}
    if op == "batch":
        w = [_solve_work(a, amg, 20, case["nrhs"]) for a, amg in _batch_plan(case["count"])]
        return {k: sum(v[k] for v in w) for k in ("bytes", "flops")}
    if op == "spmv_int":
        rptr, cind, _ = _fixed_csr(case["family"], case["side"])
        return {"bytes": 8 * len(cind) + 12 * len(rptr), "flops": 2 * len(cind)}
    a, amg = _plan_of(case)
    if op in ("vcycle", "block_vcycle"):
        return _vcycle_work(amg, case["nrhs"])
    return _solve_work(a, amg, 20 if case["family"] == "convdiff2d" else 30)


def tolerance(case):
    # every sum has a fixed order or is an integer, so results repeat bit for
    # bit; only the network's gradient adds 32-bit floats in a free order
    return {"rel": 1e-6} if case["op"] == "mlp_grad" else "exact"


def _mlp_exact(case, seed):
    w, x, t = _mlp_data(case, seed)
    w1, b1, w2, b2, w3, b3 = (v.astype(np.float64) for v in w)
    x, t = x.astype(np.float64), t.astype(np.float64)
    h1 = np.tanh(x @ w1.T + b1)
    h2 = np.tanh(h1 @ w2.T + b2)
    y = 1.0 / (1.0 + np.exp(-(h2 @ w3.T + b3)))
    d3 = 2.0 * (y - t) / len(x) * y * (1.0 - y)
    d2 = (d3 @ w3) * (1.0 - h2 * h2)
    d1 = (d2 @ w2) * (1.0 - h1 * h1)
    parts = [d1.T @ x, d1.sum(0), d2.T @ h1, d2.sum(0), d3.T @ h2, d3.sum(0)]
    return {"loss": float(((y - t) ** 2).sum() / len(x)),
            "grad": np.concatenate([v.reshape(-1) for v in parts])}


def exact(case, seed):
    if case["op"] == "mlp_grad":
        return _mlp_exact(case, seed)
    # V-cycles and the fixed-point product follow the library's own hierarchy
    # and whole numbers; the contrast of the inclusions and the unconverged
    # members of a batch leave x far from x* at this residual
    if case["op"] != "solve" or case["family"] == "inclusions3d":
        return None
    dims = 2 if case["family"].endswith("2d") else 3
    return {"x": _xstar(case["side"] ** dims, seed), "iterations": None, "status": None}
