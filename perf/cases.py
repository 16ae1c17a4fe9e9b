"""The work that a user of this library has it do, as cases that can be timed.

Each case goes through the C ABI of libomxp.so (include/omxp.h) as bench.py,
the `omxp` driver and the scheduler's training do: whole solves (generate,
factor, refine) of the three matrix families and the precision classes, and
the layers of a solve that callers use by themselves (triangular solves,
residual product, Schur update, panel step, panel solves, policy training).
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from openmxp_amd import _lib, scheduler

DEV = "cuda"
LCG_A, LCG_C = 6364136223846793005, 1
MASK64 = (1 << 64) - 1
LCG_SCALE = float.fromhex("0x1.fffffffffffffp-65")
REFLECTORS = 8  # per orthogonal factor of a randsvd matrix, as the scheduler's training and bench.py use


def listed():
    return [
        # the smallest system the tests and the smoke run solve: latency and launches
        {"name": "solve_small", "kind": "solve", "family": "lcg", "n": 1024, "b": 256, "alt": 1, "prec": "fp16",
         "method": 0},
        # the order that a CPU can factor for comparison (the bench's CPU baseline), small blocks
        {"name": "solve_fp16", "kind": "solve", "family": "lcg", "n": 10240, "b": 256, "alt": 1, "prec": "fp16",
         "method": 0},
        # the headline path (learned FP8/FP16 schedule, GMRES-IR, b = 2560) at an order whose state fits three times
        {"name": "solve_learned", "kind": "solve", "family": "lcg", "n": 61440, "b": 2560, "alt": 1,
         "prec": "learned", "method": 1},
        # a conditioned system: the FP32 Schur class with GMRES-IR, at the scheduler's training size
        {"name": "solve_randsvd", "kind": "solve", "family": "randsvd", "n": 8192, "b": 512, "alt": 1,
         "prec": "fp32", "method": 1, "kappa": 1.0e4},
        # the driver's --highammat system (kappa 1e3, rho 0.5), masked inverses (-alt 2)
        {"name": "solve_higham", "kind": "solve", "family": "higham", "n": 20480, "b": 1024, "alt": 2,
         "prec": "fp16", "method": 0, "kappa": 1.0e3},
        # one application of the factors as preconditioner: lower and upper solve
        {"name": "trsv_pair", "kind": "trsv", "n": 30720},
        # the FP64 residual with the matrix regenerated on the fly
        {"name": "residual", "kind": "residual", "n": 40960},
        # a Schur update of ragged size, FP16: pack both panels, multiply
        {"name": "schur_fp16", "kind": "schur", "fp8": False, "m": 7777, "n": 12345, "k": 2560},
        # a trailing update of a group of four panels in FP8 (k = 4 b)
        {"name": "schur_fp8", "kind": "schur", "fp8": True, "m": 20480, "n": 20480, "k": 10240},
        # the critical path of one step: diagonal block, its inverses, both panels
        {"name": "panel_step", "kind": "panel", "b": 2560, "rest": 20480},
        # the FP32 panel solves of step 0 and of -alt 0
        {"name": "panel_trsm", "kind": "trsm", "b": 2560, "rest": 30000},
        # one Adam step of the policy's training (the committed set has 2658 samples, 20000 steps)
        {"name": "policy_step", "kind": "policy", "batch": 2658},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve", "trsv", "residual", "schur", "schur", "panel", "trsm",
                       "policy"])
    if kind == "solve":
        form = rng.choice(["fp16", "learned", "randsvd", "higham"])
        top = {"learned": 40960, "randsvd": 12288}.get(form, 20480)
        b = 256 * rng.randint(*{"learned": (2, 10), "randsvd": (1, 3)}.get(form, (1, 6)))
        n = b * _log_int(rng, 3, top // b)
        if form == "learned":
            return {"kind": kind, "family": "lcg", "n": n, "b": b, "alt": rng.choice([1, 2]), "prec": "learned",
                    "method": 1}
        if form == "randsvd":
            return {"kind": kind, "family": "randsvd", "n": n, "b": b, "alt": rng.choice([0, 1]), "prec": "fp32",
                    "method": 1, "kappa": round(10 ** rng.uniform(1, 4), 2)}
        if form == "higham":
            return {"kind": kind, "family": "higham", "n": n, "b": b, "alt": rng.choice([1, 2]), "prec": "fp16",
                    "method": 0, "kappa": round(10 ** rng.uniform(2, 3), 2)}
        return {"kind": kind, "family": "lcg", "n": n, "b": b, "alt": rng.choice([0, 1, 2]), "prec": "fp16",
                "method": rng.choice([0, 1])}
    if kind == "trsv":
        return {"kind": kind, "n": _log_int(rng, 1000, 40000)}
    if kind == "residual":
        return {"kind": kind, "n": _log_int(rng, 1000, 60000)}
    if kind == "schur":
        fp8 = rng.random() < 0.5
        step = 256 if fp8 else 64
        return {"kind": kind, "fp8": fp8, "m": _log_int(rng, 500, 16000), "n": _log_int(rng, 500, 16000),
                "k": step * max(1, _log_int(rng, 256, 8192) // step)}
    if kind == "panel":
        return {"kind": kind, "b": 256 * rng.randint(1, 10), "rest": _log_int(rng, 500, 30000)}
    if kind == "trsm":
        return {"kind": kind, "b": 64 * rng.randint(4, 40), "rest": _log_int(rng, 500, 40000)}
    return {"kind": "policy", "batch": _log_int(rng, 100, 8000)}


# ---------------------------------------------------------------------------
# states and passes
# ---------------------------------------------------------------------------
def _f64(n):
    return torch.empty(n, dtype=torch.float64, device=DEV)


def _f32(n):
    return torch.empty(n, dtype=torch.float32, device=DEV)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uniform(count, g, scale=1.0, dtype=torch.float32):
    """Uniform on [-scale/2, scale/2), the generator's distribution."""
    return torch.rand(count, generator=g, dtype=dtype, device=DEV).sub_(0.5).mul_(scale)


def _bytes(count):
    return torch.empty(max(int(count), 16), dtype=torch.uint8, device=DEV)


def _pad4(n):
    return (n + 3) // 4 * 4


class _Handle:
    """A solver handle, destroyed with the state that holds it."""

    def __init__(self, n, b, alt, flags):
        self.h = C.c_void_p()
        _lib.check(_lib.lib().omx_solver_create(n, b, alt, flags, C.byref(self.h)), "solver create")

    def __del__(self):
        if self.h:
            _lib.lib().omx_solver_destroy(self.h)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["kind"]](state)


def work(case):
    return _WORK[case["kind"]](case)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


# ---- whole solves ----------------------------------------------------------
def _prepare_solve(case, seed):
    L = _lib.lib()
    n, b, prec, family = case["n"], case["b"], case["prec"], case["family"]
    learned = prec == "learned"
    s = {"kind": "solve", "case": case, "n": n, "nb": n // b, "seed": seed, "sched": None}
    s["solver"] = _Handle(n, b, case["alt"], (_lib.SOLVER_FP8 | _lib.SOLVER_GROUP4) if learned else 0)
    s["A"], s["x"], s["diag"], s["rhs"] = _f32(n * n), _f64(n), _f64(n), _f64(n)
    _lib.check(L.omx_rhs_f64(n, seed, s["rhs"].data_ptr(), None), "rhs")
    if learned:
        params = np.ascontiguousarray(scheduler.load_params())
        _lib.check(L.omx_solver_set_policy(s["solver"].h, params.ctypes.data), "policy")
    elif prec == "fp32":
        s["sched"] = np.full(s["nb"], -1, dtype=np.int32)
    if family == "lcg":
        s["system"] = _lib.System(kind=_lib.SYSTEM_LCG, seed=seed, diag=s["diag"].data_ptr())
    elif family == "randsvd":
        rank = 2 * REFLECTORS
        s["sigma"], s["P"], s["Q"], s["rowabs"] = _f64(n), _f64(n * rank), _f64(n * rank), _f64(n)
        _lib.check(L.omx_randsvd_factors(n, seed, case["kappa"], REFLECTORS, s["sigma"].data_ptr(),
                                         s["P"].data_ptr(), s["Q"].data_ptr(), None), "randsvd factors")
        s["work_bytes"] = L.omx_randsvd_workspace_bytes(n)
        s["work"] = _bytes(s["work_bytes"])
        _generate(s)
        s["system"] = _lib.System(kind=_lib.SYSTEM_LOWRANK, seed=0, diag=s["diag"].data_ptr(),
                                  norm_inf=float(s["rowabs"].max()), rank=rank, sigma=s["sigma"].data_ptr(),
                                  P=s["P"].data_ptr(), Q=s["Q"].data_ptr())
    else:
        s["alpha"], s["beta"] = _higham(n, case["kappa"])
        s["system"] = _lib.System(kind=_lib.SYSTEM_HIGHAM, seed=0, diag=s["diag"].data_ptr(),
                                  norm_inf=L.omx_higham_norm_inf(n, s["alpha"], s["beta"]), alpha=s["alpha"],
                                  beta=s["beta"])
    return s


def _higham(n, kappa):
    """(alpha, beta) of the matrix that the driver's --highammat builds."""
    rho = 0.5
    beta = _lib.lib().omx_higham_beta(n, kappa, rho)
    return -rho * beta, -beta


def _generate(s):
    L, n, family = _lib.lib(), s["n"], s["case"]["family"]
    if family == "lcg":
        rc = L.omx_matgen_f32(n, s["seed"], s["A"].data_ptr(), n, s["diag"].data_ptr(), None)
    elif family == "randsvd":
        rc = L.omx_randsvd_f32(n, 2 * REFLECTORS, s["sigma"].data_ptr(), s["P"].data_ptr(), s["Q"].data_ptr(),
                               s["A"].data_ptr(), n, s["diag"].data_ptr(), s["rowabs"].data_ptr(),
                               s["work"].data_ptr(), s["work_bytes"], None)
    else:
        rc = L.omx_higham_matgen_f32(n, s["alpha"], s["beta"], s["A"].data_ptr(), n, s["diag"].data_ptr(), None)
    _lib.check(rc, "matrix")


def _run_solve(s):
    """Generate, factor, refine; the solution and the factors."""
    L, n = _lib.lib(), s["n"]
    _generate(s)
    sched = s["sched"].ctypes.data if s["sched"] is not None else None
    _lib.check(L.omx_lu_factor(s["solver"].h, s["A"].data_ptr(), n, sched, None), "LU")
    out = np.zeros(4)
    _lib.check(L.omx_ir_solve_system(s["solver"].h, s["A"].data_ptr(), n, C.byref(s["system"]),
                                     s["rhs"].data_ptr(), s["x"].data_ptr(), s["case"]["method"], 50, 50, 1e-12,
                                     16.0, 0, out.ctypes.data, None), "refinement")
    return {"x": s["x"], "LU": s["A"]}


def _work_solve(case):
    n = float(case["n"])
    # the factors written once and read by a refinement; the LU's operations
    return {"bytes": 8.0 * n * n, "flops": 2.0 / 3.0 * n ** 3 + 1.5 * n * n}


def _exact_solve(case, seed):
    n = case["n"]
    b = _lcg_values(seed, n * n, n)
    if case["family"] == "lcg":
        if n > 24576:
            return None
        # diagonally dominant with random signs: Jacobi gains two digits a pass
        A = _lcg_matrix(n, seed)
        A.fill_diagonal_(0.0)
        d = A.abs().sum(dim=1)
        x = b / d
        for _ in range(30):
            x = (b - A @ x) / d
    elif case["family"] == "randsvd":
        # x = V diag(1/sigma) U^T b with U = H_0 .. H_{k-1}, V = H_k .. H_{2k-1}
        k = REFLECTORS
        w = [_lcg_values(seed, n * n + n + t * n, n) for t in range(2 * k)]
        w = [v / v.norm() for v in w]
        x = b.clone()
        for t in range(k):
            x = x - 2.0 * w[t] * torch.dot(w[t], x)
        i = torch.arange(n, dtype=torch.float64, device=DEV)
        x = x * case["kappa"] ** (i / (n - 1))
        for t in range(2 * k - 1, k - 1, -1):
            x = x - 2.0 * w[t] * torch.dot(w[t], x)
    else:
        # L has -alpha below, U -beta above the unit diagonal: two recurrences
        alpha, beta = _higham(n, case["kappa"])
        v, run_sum = b.cpu().numpy().astype(np.longdouble), np.longdouble(0)
        for i in range(n):
            v[i] += alpha * run_sum
            run_sum += v[i]
        run_sum = np.longdouble(0)
        for i in range(n - 1, -1, -1):
            v[i] += beta * run_sum
            run_sum += v[i]
        x = torch.from_numpy(v.astype(np.float64))
    return {"x": x, "LU": None}


# ---- the 64-bit generator, for exact() -------------------------------------
def _as_i64(v):
    v &= MASK64
    return v - (1 << 64) if v >> 63 else v


def _jump(steps):
    """The map x -> a x + c of `steps` generator steps."""
    a, c, ba, bc = 1, 0, LCG_A, LCG_C
    while steps:
        if steps & 1:
            a, c = a * ba & MASK64, (a * bc + c) & MASK64
        ba, bc = ba * ba & MASK64, (ba * bc + bc) & MASK64
        steps >>= 1
    return a, c


def _maps(count, stride):
    """The maps of 0, stride, 2 stride, ... steps, as two int64 tensors."""
    a = torch.ones(1, dtype=torch.int64, device=DEV)
    c = torch.zeros(1, dtype=torch.int64, device=DEV)
    while a.numel() < count:
        ja, jc = _jump(stride * a.numel())
        a, c = torch.cat([a, a * _as_i64(ja)]), torch.cat([c, c * _as_i64(ja) + _as_i64(jc)])
    return a[:count], c[:count]


def _states(seed, first, count):
    x0 = (LCG_A * seed + LCG_C) & MASK64
    ja, jc = _jump(first)
    a, c = _maps(count, 1)
    return a * _as_i64((ja * x0 + jc) & MASK64) + c


def _lcg_values(seed, first, count):
    return _states(seed, first, count).double() * LCG_SCALE


def _lcg_rows(n, seed, i0, i1):
    """Rows i0 .. i1 of the order-n matrix (element (i, j) has index i + n j), no diagonal substitution."""
    a, c = _maps(n, n)
    s = _states(seed, i0, i1 - i0)
    return (s[:, None] * a[None, :] + c[None, :]).double() * LCG_SCALE


def _lcg_matrix(n, seed):
    return torch.cat([_lcg_rows(n, seed, i, min(n, i + 2048)) for i in range(0, n, 2048)])


# ---- triangular solves -----------------------------------------------------
def _prepare_trsv(case, seed):
    """Factors as the LU of a diagonally dominant system leaves them, and a residual."""
    L, n = _lib.lib(), case["n"]
    g, lda = _gen(seed), _pad4(case["n"])
    A = _uniform(n * lda, g).view(n, lda)  # A[j, i]: column j
    for j in range(0, n, 2048):
        cols = torch.arange(j, min(n, j + 2048), device=DEV)[:, None]
        below = torch.arange(lda, device=DEV)[None, :] > cols
        A[j:j + 2048].mul_(torch.where(below, 4.0 / n, 1.0))
    A.diagonal().copy_(n / 4.0 * (1.0 + 0.05 * _uniform(n, g)))
    wb = L.omx_trsv_workspace_bytes(n)
    return {"kind": "trsv", "n": n, "lda": lda, "A": A, "r": _uniform(n, g, dtype=torch.float64), "x": _f64(n),
            "work": _bytes(wb), "work_bytes": wb}


def _run_trsv(s):
    L, n = _lib.lib(), s["n"]
    wp = s["work"].data_ptr() if s["work_bytes"] else None
    _lib.check(L.omx_copy_f64(n, s["r"].data_ptr(), s["x"].data_ptr(), None), "copy")
    _lib.check(L.omx_trsv_lower_unit_f32f64(n, n, s["A"].data_ptr(), s["lda"], s["x"].data_ptr(), wp,
                                            s["work_bytes"], None), "lower solve")
    _lib.check(L.omx_trsv_upper_f32f64(n, n, s["A"].data_ptr(), s["lda"], s["x"].data_ptr(), wp, s["work_bytes"],
                                       None), "upper solve")
    return s["x"]


def _work_trsv(case):
    n = float(case["n"])
    return {"bytes": 4.0 * n * n, "flops": 2.0 * n * n}


def _exact_trsv(case, seed):
    s = _prepare_trsv(case, seed)
    n = s["n"]
    A = s["A"][:, :n].double().t()
    y = torch.linalg.solve_triangular(A, s["r"][:, None], upper=False, unitriangular=True)
    return torch.linalg.solve_triangular(A, y, upper=True)[:, 0]


# ---- residual --------------------------------------------------------------
def _prepare_residual(case, seed):
    L, n = _lib.lib(), case["n"]
    g = _gen(seed)
    diag = _f64(n)
    _lib.check(L.omx_diag_f64(n, seed, 0, n, diag.data_ptr(), None), "diagonal")
    wb = L.omx_otf_gemv_workspace_bytes(n)
    b = _uniform(n, g, dtype=torch.float64)
    return {"kind": "residual", "n": n, "seed": seed, "diag": diag, "b": b, "r": _f64(n),
            "x": _uniform(n, g, 4.0 / n, dtype=torch.float64), "work": _bytes(wb), "work_bytes": wb,
            "norm": _f64(1)}


def _run_residual(s):
    """r = b - A x and its norm, as one refinement step forms them."""
    L, n = _lib.lib(), s["n"]
    wp = s["work"].data_ptr() if s["work_bytes"] else None
    _lib.check(L.omx_copy_f64(n, s["b"].data_ptr(), s["r"].data_ptr(), None), "copy")
    _lib.check(L.omx_otf_gemv_f64(n, s["seed"], s["diag"].data_ptr(), -1.0, s["x"].data_ptr(), s["r"].data_ptr(),
                                  wp, s["work_bytes"], None), "residual")
    _lib.check(L.omx_norm_inf_f64(n, s["r"].data_ptr(), s["norm"].data_ptr(), None), "norm")
    return {"r": s["r"], "norm": s["norm"]}


def _work_residual(case):
    n = float(case["n"])
    return {"bytes": 40.0 * n, "flops": 2.0 * n * n}


def _exact_residual(case, seed):
    n = case["n"]
    g = _gen(seed)
    b = _uniform(n, g, dtype=torch.float64)
    x = _uniform(n, g, 4.0 / n, dtype=torch.float64)
    out = []
    for i in range(0, n, 1024):
        i1 = min(n, i + 1024)
        R = _lcg_rows(n, seed, i, i1)
        rows = torch.arange(i1 - i, device=DEV)
        R[rows, rows + i] = 0.0
        R[rows, rows + i] = R.abs().sum(dim=1)
        out.append(b[i:i1] - R @ x)
    r = torch.cat(out)
    return {"r": r, "norm": r.abs().max()[None]}


# ---- Schur update ----------------------------------------------------------
def _schur_inputs(case, seed):
    g, m, n, k = _gen(seed), case["m"], case["n"], case["k"]
    scale = 4.0 / max(m, n, k)  # column panels are divided by the pivots
    return _uniform(k * m, g, scale).view(k, m), _uniform(n * k, g).view(n, k), _uniform(n * m, g).view(n, m)


def _prepare_schur(case, seed):
    L, m, n, k, fp8 = _lib.lib(), case["m"], case["n"], case["k"], case["fp8"]
    col, row, Cm = _schur_inputs(case, seed)
    s = {"kind": "schur", "case": case, "col": col, "row": row, "C": Cm,
         "X": _bytes(L.omx_panel_bytes(m, k, int(fp8))), "Y": _bytes(L.omx_panel_bytes(n, k, int(fp8)))}
    if fp8:
        for name, rows in (("X", m), ("Y", n)):
            count = L.omx_panel_exps_count(rows, k)
            s[name + "e"] = torch.empty(count, dtype=torch.int32, device=DEV)
            s[name + "m"] = _f32(count)
    return s


def _run_schur(s):
    """C -= col row: both panels packed, one product."""
    L, c = _lib.lib(), s["case"]
    m, n, k = c["m"], c["n"], c["k"]
    col, row, X, Y, Cm = (s[v].data_ptr() for v in ("col", "row", "X", "Y", "C"))
    if c["fp8"]:
        Xe, Xm, Ye, Ym = (s[v].data_ptr() for v in ("Xe", "Xm", "Ye", "Ym"))
        _lib.check(L.omx_pack_f8(m, k, col, 1, m, X, Xe, Xm, None), "pack column panel")
        _lib.check(L.omx_pack_f8(n, k, row, k, 1, Y, Ye, Ym, None), "pack row panel")
        _lib.check(L.omx_gemm_f8_packed(m, n, k, -1.0, X, Xe, 0, Y, Ye, 0, 1.0, Cm, m, None), "product")
    else:
        _lib.check(L.omx_pack_f16(m, k, col, 1, m, _MASK_NONE, X, None, None), "pack column panel")
        _lib.check(L.omx_pack_f16(n, k, row, k, 1, _MASK_NONE, Y, None, None), "pack row panel")
        _lib.check(L.omx_gemm_f16_packed(m, n, k, -1.0, X, 0, Y, 0, 1.0, Cm, m, None), "product")
    return s["C"]


def _work_schur(case):
    m, n, k = float(case["m"]), float(case["n"]), float(case["k"])
    return {"bytes": 8.0 * m * n + 4.0 * (m + n) * k, "flops": 2.0 * m * n * k}


def _quantised(S, fp8):
    """rows x k panel as the products see it, in 64 bits."""
    if not fp8:
        return S.half().double()
    rows, k = S.shape
    out = torch.empty_like(S, dtype=torch.float64)
    for r in range(0, rows, 256):
        for c in range(0, k, 256):
            t = S[r:r + 256, c:c + 256]
            fm, em = torch.frexp(t.abs().max())
            e = torch.where(fm <= 0.875, 9 - em, 8 - em).double()
            scale = torch.exp2(e)
            q = (t * scale.float()).to(torch.float8_e4m3fn)
            out[r:r + 256, c:c + 256] = q.float().double() / scale
    return out


def _exact_schur(case, seed):
    col, row, Cm = _schur_inputs(case, seed)
    X = _quantised(col.t().contiguous(), case["fp8"])
    Y = _quantised(row, case["fp8"])
    return Cm.double().sub_(Y @ X.t().contiguous())  # column-major: the transpose


# ---- panel step ------------------------------------------------------------
_MASK_NONE = 0
_RUNN, _LLNU = 0, 1


def _panel_inputs(b, rest, seed):
    """Column panel [D; below] (ld = b + rest, padded) and row panel (ld = b) of a diagonally dominant step."""
    g, ld = _gen(seed), _pad4(b + rest)
    col = _uniform(b * ld, g).view(b, ld)
    col[:, :b].diagonal().copy_((b + rest) / 4.0 * (1.0 + 0.05 * _uniform(b, g)))
    return ld, col, _uniform(rest * b, g).view(rest, b)


def _prepare_panel(case, seed):
    L, b, rest = _lib.lib(), case["b"], case["rest"]
    ld, col, row = _panel_inputs(b, rest, seed)
    s = {"kind": "panel", "b": b, "rest": rest, "ld": ld, "col0": col, "row0": row,
         "col": torch.empty_like(col), "row": torch.empty_like(row)}
    for name in ("Xu", "Xl", "W"):
        s[name] = _f32(b * b)
    s["Uh"], s["Lh"] = _bytes(L.omx_panel_bytes(b, b, 0)), _bytes(L.omx_panel_bytes(b, b, 0))
    s["T"] = _bytes(L.omx_panel_bytes(rest, b, 0))
    s["info"] = torch.empty(1, dtype=torch.int32, device=DEV)
    tiles = L.omx_panel_exps_count(rest, b)
    s["lmax"], s["rmax"] = _f32(tiles), _f32(tiles)
    return s


def _run_panel(s):
    """getrf of the diagonal block, its inverses, the FP16 inverse products of both panels and their tile maxima."""
    L, b, rest, ld = _lib.lib(), s["b"], s["rest"], s["ld"]
    ck = _lib.check
    col, row, Xu, Xl, W, Uh, Lh, T = (s[v].data_ptr() for v in ("col", "row", "Xu", "Xl", "W", "Uh", "Lh", "T"))
    below = col + 4 * b
    ck(L.omx_copy_block_f32(b + rest, b, s["col0"].data_ptr(), ld, col, ld, None), "copy")
    ck(L.omx_copy_block_f32(b, rest, s["row0"].data_ptr(), b, row, b, None), "copy")
    ck(L.omx_getrf_nopiv_f32(b, col, ld, s["info"].data_ptr(), None), "getrf")
    ck(L.omx_trtri_lu_f32(b, col, ld, Xu, Xl, b, W, None), "inverses")
    ck(L.omx_pack_f16(b, b, Xu, b, 1, _MASK_NONE, Uh, None, None), "pack")
    ck(L.omx_pack_f16(rest, b, below, 1, ld, _MASK_NONE, T, None, None), "pack")
    ck(L.omx_gemm_f16_packed_tri(rest, b, b, 1.0, T, Uh, 1, 0.0, below, ld, s["lmax"].data_ptr(), None), "column")
    ck(L.omx_pack_f16(b, b, Xl, 1, b, _MASK_NONE, Lh, None, None), "pack")
    ck(L.omx_pack_f16(rest, b, row, b, 1, _MASK_NONE, T, None, None), "pack")
    ck(L.omx_gemm_f16_packed_tri(b, rest, b, 1.0, Lh, T, 2, 0.0, row, b, s["rmax"].data_ptr(), None), "row")
    return {"col": s["col"][:, :b + rest], "row": s["row"], "info": s["info"], "lmax": s["lmax"],
            "rmax": s["rmax"]}


def _work_panel(case):
    b, r = float(case["b"]), float(case["rest"])
    return {"bytes": 8.0 * (b * b + 2.0 * r * b), "flops": 2.0 / 3.0 * b ** 3 + 2.0 * r * b * b}


def _lu_nopivot(D):
    D = D.clone()
    n = D.shape[0]
    for j in range(0, n, 64):
        e = min(n, j + 64)
        for k in range(j, e):
            D[k + 1:, k] /= D[k, k]
            D[k + 1:, k + 1:e] -= D[k + 1:, k:k + 1] * D[k:k + 1, k + 1:e]
        if e < n:
            D[j:e, e:] = torch.linalg.solve_triangular(D[j:e, j:e], D[j:e, e:], upper=False, unitriangular=True)
            D[e:, e:] -= D[e:, j:e] @ D[j:e, e:]
    return D


def _exact_panel(case, seed):
    b, rest = case["b"], case["rest"]
    _, col, row = _panel_inputs(b, rest, seed)
    A = col[:, :b + rest].double()  # A[j, i]: column j
    D = _lu_nopivot(A[:, :b].t().contiguous())
    below = torch.linalg.solve_triangular(D.t(), A[:, b:], upper=False)  # U^T (L21^T) = A21^T
    right = torch.linalg.solve_triangular(D, row.double().t(), upper=False, unitriangular=True)
    return {"col": torch.cat([D.t(), below], dim=1), "row": right.t().contiguous(), "info": None, "lmax": None,
            "rmax": None}


# ---- FP32 panel solves -----------------------------------------------------
def _trsm_inputs(case, seed):
    """A factored diagonal block (ld = b) and the two panels (ld padded, and b)."""
    b, rest = case["b"], case["rest"]
    g, ld = _gen(seed), _pad4(rest)
    n = b + rest
    T = _uniform(b * b, g).view(b, b)  # T[j, i]: column j
    T.mul_(torch.where(torch.ones_like(T, dtype=torch.bool).triu(1), 4.0 / n, 1.0))
    T.diagonal().copy_(n / 4.0 * (1.0 + 0.05 * _uniform(b, g)))
    return T, ld, _uniform(b * ld, g).view(b, ld), _uniform(rest * b, g).view(rest, b)


def _prepare_trsm(case, seed):
    T, ld, col, row = _trsm_inputs(case, seed)
    return {"kind": "trsm", "b": case["b"], "rest": case["rest"], "ld": ld, "T": T, "col0": col, "row0": row,
            "col": torch.empty_like(col), "row": torch.empty_like(row)}


def _run_trsm(s):
    L, b, rest, ld = _lib.lib(), s["b"], s["rest"], s["ld"]
    T, col, row = (s[v].data_ptr() for v in ("T", "col", "row"))
    _lib.check(L.omx_copy_block_f32(rest, b, s["col0"].data_ptr(), ld, col, ld, None), "copy")
    _lib.check(L.omx_copy_block_f32(b, rest, s["row0"].data_ptr(), b, row, b, None), "copy")
    _lib.check(L.omx_trsm_f32(_RUNN, rest, b, T, b, col, ld, None), "column panel")
    _lib.check(L.omx_trsm_f32(_LLNU, b, rest, T, b, row, b, None), "row panel")
    return {"col": s["col"][:, :rest], "row": s["row"]}


def _work_trsm(case):
    b, r = float(case["b"]), float(case["rest"])
    return {"bytes": 4.0 * b * b + 16.0 * r * b, "flops": 2.0 * r * b * b}


def _exact_trsm(case, seed):
    T, _, col, row = _trsm_inputs(case, seed)
    T = T.double()  # T[j, i] = block(i, j)
    c = torch.linalg.solve_triangular(T, col[:, :case["rest"]].double(), upper=False)  # U^T X^T = B^T
    r = torch.linalg.solve_triangular(T.t(), row.double().t(), upper=False, unitriangular=True)
    return {"col": c, "row": r.t().contiguous()}


# ---- policy training -------------------------------------------------------
_LR, _B1, _B2, _EPS, _STEP = 3e-3, 0.9, 0.999, 1e-8, 500


def _policy_inputs(case, seed):
    """Features, labels, headroom targets and masks of a batch; parameters and moments in mid-training."""
    g, batch = _gen(seed), case["batch"]
    X = torch.randn(batch, scheduler.NFEAT, generator=g, device=DEV).mul_(0.6)
    y = (torch.rand(batch, generator=g, device=DEV) < 0.73).to(torch.int32)
    t = (torch.rand(batch, generator=g, device=DEV) < 0.2).float()
    P = torch.from_numpy(scheduler.init_params(seed)).to(DEV)
    mom = torch.randn(scheduler.NPARAMS, generator=g, device=DEV).mul_(1e-3)
    vel = torch.rand(scheduler.NPARAMS, generator=g, device=DEV).add_(0.5).mul_(1e-4)
    return X, y, t, y.float(), P, mom, vel


def _prepare_policy(case, seed):
    L, batch = _lib.lib(), case["batch"]
    s = dict(zip(("X", "y", "t", "m", "P", "mom", "vel"), _policy_inputs(case, seed)))
    wb = L.omx_mlp_backward_workspace_bytes(batch)
    s.update(kind="policy", batch=batch, H1=_f32(batch * 64), H2=_f32(batch * 64), Z=_f32(batch * 3),
             G=_f32(scheduler.NPARAMS), loss=_f32(1), work=_bytes(wb), work_bytes=wb, step=_STEP)
    return s


def _run_policy(s):
    """Forward, backward and Adam update, as scheduler.train runs them."""
    L, batch = _lib.lib(), s["batch"]
    P, X, H1, H2, Z, G = (s[v].data_ptr() for v in ("P", "X", "H1", "H2", "Z", "G"))
    _lib.check(L.omx_mlp_forward_f32(batch, P, X, H1, H2, Z, None), "forward")
    _lib.check(L.omx_mlp_backward_f32(batch, P, X, H1, H2, Z, s["y"].data_ptr(), s["t"].data_ptr(),
                                      s["m"].data_ptr(), G, s["loss"].data_ptr(), s["work"].data_ptr(),
                                      s["work_bytes"], None), "backward")
    _lib.check(L.omx_mlp_adam_f32(scheduler.NPARAMS, P, G, s["mom"].data_ptr(), s["vel"].data_ptr(), _LR, _B1, _B2,
                                  _EPS, s["step"], None), "adam")
    s["step"] += 1
    return {"Z": s["Z"], "grad": s["G"], "loss": s["loss"], "P": s["P"], "mom": s["mom"], "vel": s["vel"]}


def _work_policy(case):
    # forward, gradients of the layers' inputs and of their weights; activations and deltas written once
    mac = scheduler.NFEAT * 64 + 64 * 64 + 64 * 3
    return {"bytes": case["batch"] * 4.0 * (scheduler.NFEAT + 131 + 131 + 3) + 4.0 * 7 * scheduler.NPARAMS,
            "flops": 6.0 * mac * case["batch"]}


def _exact_policy(case, seed):
    X, y, t, m, P, mom, vel = (v.double() for v in _policy_inputs(case, seed))
    P0, P = P, P.clone().requires_grad_()
    W1, b1, W2, b2, W3, b3 = torch.split(P, [16 * 64, 64, 64 * 64, 64, 64 * 3, 3])
    h1 = torch.relu(X @ W1.view(16, 64) + b1)
    h2 = torch.relu(h1 @ W2.view(64, 64) + b2)
    z = h2 @ W3.view(64, 3) + b3
    loss = torch.nn.functional.cross_entropy(z[:, :2], y.long()) + (0.5 * m * (z[:, 2] - t) ** 2).mean()
    loss.backward()
    G = P.grad
    mom = _B1 * mom + (1 - _B1) * G
    vel = _B2 * vel + (1 - _B2) * G * G
    P1 = P0 - _LR * (mom / (1 - _B1 ** _STEP)) / ((vel / (1 - _B2 ** _STEP)).sqrt() + _EPS)
    return {"Z": z.detach().reshape(-1), "grad": G, "loss": loss.detach()[None], "P": P1, "mom": mom, "vel": vel}


_PREPARE = {"solve": _prepare_solve, "trsv": _prepare_trsv, "residual": _prepare_residual, "schur": _prepare_schur,
            "panel": _prepare_panel, "trsm": _prepare_trsm, "policy": _prepare_policy}
_RUN = {"solve": _run_solve, "trsv": _run_trsv, "residual": _run_residual, "schur": _run_schur,
        "panel": _run_panel, "trsm": _run_trsm, "policy": _run_policy}
_WORK = {"solve": _work_solve, "trsv": _work_trsv, "residual": _work_residual, "schur": _work_schur,
         "panel": _work_panel, "trsm": _work_trsm, "policy": _work_policy}
_EXACT = {"solve": _exact_solve, "trsv": _exact_trsv, "residual": _exact_residual, "schur": _exact_schur,
          "panel": _exact_panel, "trsm": _exact_trsm, "policy": _exact_policy}
