"""The work that a user of this library has it do, as cases that can be timed and checked.

Eight forms, each through the public entry points of the `hplai` binding:

  solve      Context.solve: generate, factor, refine, read x back
  autograd   hplai.autograd.solve and its backward: X, dA, dB
  batch      Batch.run("graph") over many small systems, every solution read back
  residual   Context.otf_gemv: the matrix-free FP64 residual
  generate   Context.gen_diag, gen_rhs and gen_matrix of a whole matrix
  panel      Context.getrf, trsm_lpanel and trsm_upanel of one block step
  update     Context.quantize of a K-slice stack of panels, then schur_update
  gemmschur  Context.gemmschur_f16 with the reference's operand layout

Matrices follow the HPL-AI rules throughout: off-diagonal entries uniform in
[-0.5, 0.5), a diagonal that is the row's sum of magnitudes, factors of the
sizes that an LU of such a matrix has.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hpl-ai_amd"))

import hplai  # noqa: E402
from hplai import autograd  # noqa: E402

DEV = "cuda"
LCG_A = 6364136223846793005
SCALE = float.fromhex("0x1.fffffffffffffp-65")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the reference's own small run (n = 1200, b = 60, FP16): a few milliseconds, all latency
        dict(name="solve_1200_b60_f16", form="solve", n=1200, b=60, fmt="f16", outer=1, lazy=0),
        # the size the parity tests use with every format: one diagonal block in sixteen
        dict(name="solve_8192_b512_e4m3", form="solve", n=8192, b=512, fmt="e4m3", outer=4, lazy=0),
        # the mid-size configuration (n = 61440, FP16 Schur update)
        dict(name="solve_61440_b512_f16", form="solve", n=61440, b=512, fmt="f16", outer=16, lazy=0),
        # the benchmark's schedule (e4m3, outer 16) at half its order
        dict(name="solve_98304_b512_e4m3", form="solve", n=98304, b=512, fmt="e4m3", outer=16, lazy=0),
        # the differentiable solve at its benchmark size, forward and backward
        dict(name="autograd_8192x64", form="autograd", n=8192, k=64, b=512, fmt="f16", outer=1),
        # the same for a small system with few right-hand sides (a layer of a larger model)
        dict(name="autograd_1200x3", form="autograd", n=1200, k=3, b=60, fmt="f16", outer=1),
        # serving many small systems of uneven sizes
        dict(name="batch_1024", form="batch", count=1024, nmin=32, nmax=1024),
        # one refinement residual of the mid-size configuration
        dict(name="residual_61440", form="residual", n=61440),
        # a matrix generated for a caller's own solver, of odd order
        dict(name="generate_10007", form="generate", n=10007),
        # one block step's panel work bound from a caller's own LU
        dict(name="panel_512x40000", form="panel", b=512, m=40000, n=40000),
        # one trailing update of the benchmark's schedule from FP32 panels (16 slices of 512)
        dict(name="update_32768x8192_e4m3", form="update", m=32768, n=32768, b=512, slices=16, fmt="e4m3"),
        # the reference's Schur seam at a ragged local shape with its K = b = 60
        dict(name="gemmschur_4001x3003x60", form="gemmschur", n=4001, m=3003, k=60),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    form = rng.choice(["solve", "solve", "autograd", "autograd", "batch", "residual", "generate", "panel", "update",
                       "gemmschur"])
    if form == "solve":
        fmt = rng.choice(["f16", "e4m3", "f16t"])
        b = rng.choice([128, 256, 512]) if fmt != "f16" else rng.choice([60, 100, 128, 256, 512])
        blocks = max(2, _log(rng, 1200, 120 * b) // b)      # small blocks go with small orders
        return dict(form=form, n=b * blocks, b=b, fmt=fmt, outer=rng.choice([1, 4, 8, 16]),
                    lazy=rng.choice([0, 0, 0, 1]))
    if form == "autograd":
        fmt = rng.choice(["f16", "f16", "e4m3"])
        b = rng.choice([128, 256, 512]) if fmt == "e4m3" else rng.choice([60, 100, 128, 256, 512])
        blocks = max(2, _log(rng, 1000, 8192) // b)
        return dict(form=form, n=b * blocks, k=_log(rng, 1, 96), b=b, fmt=fmt, outer=rng.choice([1, 1, 4]))
    if form == "batch":
        nmin = _log(rng, 2, 256)
        return dict(form=form, count=_log(rng, 32, 1024), nmin=nmin, nmax=min(1024, nmin + _log(rng, 16, 1024)))
    if form == "residual":
        return dict(form=form, n=_log(rng, 1000, 61440))
    if form == "generate":
        return dict(form=form, n=_log(rng, 500, 24000))
    if form == "panel":
        return dict(form=form, b=rng.choice([60, 100, 128, 256, 320, 512, 777, 1000]), m=_log(rng, 500, 40000),
                    n=_log(rng, 500, 40000))
    if form == "update":
        b = rng.choice([128, 256, 512])
        return dict(form=form, m=_log(rng, 500, 24000), n=_log(rng, 500, 24000), b=b,
                    slices=_log(rng, 1, 4096 // b), fmt=rng.choice(["f16", "f16t", "e4m3", "e4m3"]))
    return dict(form=form, n=_log(rng, 300, 16000), m=_log(rng, 300, 16000), k=_log(rng, 32, 1024))


def work(case):
    f = case["form"]
    if f == "solve":
        # the factors are written once and read once by the triangular solves
        n = case["n"]
        return dict(bytes=8.0 * n * n, flops=2.0 / 3.0 * n ** 3 + 1.5 * n * n)
    if f == "autograd":
        # A, B, W in, X, dA, dB out; one LU, two solves and the gradient's product
        n, k = case["n"], case["k"]
        return dict(bytes=16.0 * n * n + 32.0 * n * k, flops=2.0 / 3.0 * n ** 3 + 6.0 * n * n * k)
    if f == "batch":
        n, r, _ = _batch(case, 0)
        n = n.astype(np.float64)
        return dict(bytes=float((8.0 * n * n + 8.0 * n * r).sum()), flops=float((2.0 / 3.0 * n ** 3).sum()))
    if f == "residual":
        n = case["n"]
        return dict(bytes=32.0 * n, flops=2.0 * n * n)
    if f == "generate":
        n = case["n"]
        return dict(bytes=4.0 * n * n + 16.0 * n, flops=1.0 * n * n)
    if f == "panel":
        b, m, n = case["b"], case["m"], case["n"]
        return dict(bytes=8.0 * b * (b + m + n), flops=2.0 / 3.0 * b ** 3 + 1.0 * (m + n) * b * b)
    if f == "update":
        m, n, k = case["m"], case["n"], case["b"] * case["slices"]
        es = 1 if case["fmt"] == "e4m3" else 2
        return dict(bytes=(4.0 + es) * (m + n) * k + 8.0 * m * n, flops=2.0 * m * n * k)
    n, m, k = case["n"], case["m"], case["k"]
    return dict(bytes=2.0 * (n + m) * k + 8.0 * n * m, flops=2.0 * n * m * k)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _uniform(shape, g, dtype, scale=1.0):
    """Uniform in [-scale / 2, scale / 2)."""
    return torch.rand(shape, generator=g, dtype=dtype, device=DEV).sub_(0.5).mul_(scale)


def _batch(case, seed):
    """Sizes and numbers of right-hand sides belong to the case, the matrices to the seed."""
    rng = np.random.default_rng(2024)
    n = rng.integers(case["nmin"], case["nmax"] + 1, size=case["count"]).astype(np.int32)
    nrhs = rng.integers(1, 5, size=case["count"]).astype(np.int32)
    seeds = np.random.default_rng(seed).integers(1, 2 ** 62, size=case["count"], dtype=np.int64).astype(np.uint64)
    return n, nrhs, seeds


def _dense(n, k, seed):
    """A of the HPL-AI kind in FP64, B and W with k columns."""
    g = _gen(seed)
    A = _uniform((n, n), g, torch.float64)
    A.diagonal().zero_()
    A.diagonal().copy_(A.abs().sum(1))
    return A, _uniform((n, k), g, torch.float64), _uniform((n, k), g, torch.float64)


def _panel(case, seed):
    """Diagonal block (b x b), the rows below (m x b) and the block row (b x n), column-major."""
    b, m, n = case["b"], case["m"], case["n"]
    g = _gen(seed)
    D = _uniform((b, b), g, torch.float32)
    D.diagonal().copy_(0.25 * (b + m) + _uniform((b,), g, torch.float32))
    return D, _uniform((b, m), g, torch.float32), _uniform((n, b), g, torch.float32)


def _update(case, seed):
    """L panel (m x K, entries of about 2 / n), U panel (K x n) and C (m x n), column-major."""
    m, n, k = case["m"], case["n"], case["b"] * case["slices"]
    g = _gen(seed)
    L = _uniform((k, m), g, torch.float32, 4.0 / (m + k))
    U = _uniform((n, k), g, torch.float32)
    return L, U, _uniform((n, m), g, torch.float32)


def _seam(case, seed):
    n, m, k = case["n"], case["m"], case["k"]
    g = _gen(seed)
    a = _uniform((k, n), g, torch.float32, 4.0 / (n + k)).half()
    b = _uniform((m, k), g, torch.float32).half()
    return a, b, _uniform((m, n), g, torch.float32)


def prepare(case, seed):
    f = case["form"]
    ctx = hplai.Context(0)
    s = dict(case=case, ctx=ctx, seed=int(seed))
    if f == "autograd":
        A, B, W = _dense(case["n"], case["k"], seed)
        s.update(A=A.requires_grad_(), B=B.requires_grad_(), W=W)
    elif f == "batch":
        s["batch"] = hplai.Batch(ctx, *_batch(case, seed))
        s["batch"].autotune()
    elif f == "residual":
        n = case["n"]
        g = _gen(seed)
        d = torch.empty(n, dtype=torch.float64, device=DEV)
        ctx.gen_diag(n, s["seed"], 0, n, d)
        # x as the refinement has it: right-hand side over diagonal
        rhs = _uniform((n,), g, torch.float64)
        s.update(d=d, rhs=rhs, x=rhs / d, y=torch.empty_like(rhs))
    elif f == "generate":
        n = case["n"]
        s.update(A=torch.empty((n, n), dtype=torch.float32, device=DEV),
                 d=torch.empty(n, dtype=torch.float64, device=DEV),
                 b=torch.empty(n, dtype=torch.float64, device=DEV))
    elif f == "panel":
        D, L, U = _panel(case, seed)
        s.update(inputs=(D, L, U), outs=tuple(torch.empty_like(t) for t in (D, L, U)),
                 info=torch.zeros(1, dtype=torch.int32, device=DEV))
    elif f == "update":
        L, U, C = _update(case, seed)
        m, n, b, sl = case["m"], case["n"], case["b"], case["slices"]
        qt = torch.uint8 if case["fmt"] == "e4m3" else torch.int16
        s.update(L=L, U=U, C=C, Lq=torch.empty((m, b * sl), dtype=qt, device=DEV),
                 Uq=torch.empty((n, b * sl), dtype=qt, device=DEV),
                 eL=torch.empty((sl, -(-m // b)), dtype=torch.int32, device=DEV),
                 eU=torch.empty((sl, -(-n // b)), dtype=torch.int32, device=DEV))
    elif f == "gemmschur":
        a, b, c = _seam(case, seed)
        s.update(a=a, b=b, c=c)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    case, ctx = s["case"], s["ctx"]
    f = case["form"]
    if f == "solve":
        n, lazy = case["n"], bool(case["lazy"])
        # lazy initialisation with the 16-bit partial sums where the library takes them, as the driver's -d
        trail16 = lazy and case["b"] % 128 == 0 and case["fmt"] != "f16t"
        r = ctx.solve(n, case["b"], fmt=case["fmt"], outer=case["outer"], seed=s["seed"], lazy=lazy, trail16=trail16,
                      keep_factors=True)
        x = ctx.solution_x(n)
        ctx.release()
        return dict(x=x, converged=r["converged"])
    if f == "autograd":
        X = autograd.solve(s["A"], s["B"], ctx=ctx, b=case["b"], fmt=case["fmt"], outer=case["outer"])
        dA, dB = torch.autograd.grad(X, (s["A"], s["B"]), s["W"])
        return dict(X=X.detach(), dA=dA, dB=dB)
    if f == "batch":
        bt = s["batch"]
        bt.run("graph")
        _, _, info, _ = bt.results()
        return dict(x=np.concatenate([bt.solution(q).T.ravel() for q in range(bt.count)]), info=info)
    if f == "residual":
        s["y"].copy_(s["rhs"])
        ctx.otf_gemv(case["n"], s["seed"], s["d"], -1.0, s["x"], s["y"])
        return s["y"]
    if f == "generate":
        n = case["n"]
        ctx.gen_diag(n, s["seed"], 0, n, s["d"])
        ctx.gen_rhs(n, s["seed"], 0, n, s["b"])
        ctx.gen_matrix(n, s["seed"], 0, 0, n, n, s["d"], s["A"], n)
        return dict(A=s["A"], d=s["d"], b=s["b"])
    if f == "panel":
        b, m, n = case["b"], case["m"], case["n"]
        D, L, U = s["outs"]
        for o, i in zip(s["outs"], s["inputs"]):
            o.copy_(i)
        ctx.getrf(b, D, b, s["info"])
        ctx.trsm_lpanel(m, b, D, b, L, m)
        ctx.trsm_upanel(b, n, D, b, U, b)
        return dict(D=D, L=L, U=U, info=s["info"])
    if f == "update":
        m, n, b, sl = case["m"], case["n"], case["b"], case["slices"]
        K, code = b * sl, hplai.FMTS[case["fmt"]]
        L, U, Lq, Uq, eL, eU, C = (s[q] for q in ("L", "U", "Lq", "Uq", "eL", "eU", "C"))
        tiled = case["fmt"] != "f16"
        for t in range(sl):
            ctx.quantize(code, 0, m, b, b, L[t * b:], m, Lq[:, t * b:], K, eL[t] if tiled else None)
            ctx.quantize(code, 1, n, b, b, U[:, t * b:], K, Uq[:, t * b:], K, eU[t] if tiled else None)
        ctx.schur_update(code, m, n, sl, b, Lq, K, eL if tiled else None, eL.shape[1], Uq, K, eU if tiled else None,
                         eU.shape[1], b, C, m)
        out = dict(C=C, Lq=Lq, Uq=Uq)
        if tiled:
            out.update(eL=eL, eU=eU)
        return out
    n, m, k = case["n"], case["m"], case["k"]
    ctx.gemmschur_f16(n, m, k, s["a"], n, s["b"], k, s["c"], n)
    return s["c"]


# ---------------------------------------------------------------------------
# the same in 64 bits with plain torch
# ---------------------------------------------------------------------------
def _wrap(v):
    """A Python integer as the int64 of the same low 64 bits."""
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def _lcg_powers(a, c, count):
    """(a_k, c_k) of k steps of x -> a x + c mod 2^64 for k = 0 .. count - 1."""
    A = torch.ones(1, dtype=torch.int64, device=DEV)
    C = torch.zeros(1, dtype=torch.int64, device=DEV)
    am, cm = a, c                                        # the map of A.numel() steps
    while A.numel() < count:
        C = torch.cat([C, A * _wrap(cm) + C])
        A = torch.cat([A, A * _wrap(am)])
        am, cm = am * am, am * cm + cm
        am, cm = am & ((1 << 64) - 1), cm & ((1 << 64) - 1)
    return A[:count], C[:count]


def _lcg_step(count):
    """(a, c) of `count` steps."""
    a, c, ra, rc = LCG_A, 1, 1, 0
    mask = (1 << 64) - 1
    while count:
        if count & 1:
            ra, rc = a * ra & mask, (a * rc + c) & mask
        a, c = a * a & mask, (a * c + c) & mask
        count >>= 1
    return ra, rc


def _lcg_matrix(n, seed, extra=0):
    """(n + extra, n): column j of the stream's n x (n + extra) array at row j, in FP64."""
    rows = _lcg_powers(LCG_A, 1, n)
    cols = _lcg_powers(*_lcg_step(n), n + extra)
    x1 = _wrap(LCG_A * seed + 1)
    M = torch.empty((n + extra, n), dtype=torch.float64, device=DEV)
    for j in range(0, n + extra, 2048):
        s0 = cols[0][j:j + 2048] * x1 + cols[1][j:j + 2048]
        M[j:j + 2048] = (s0[:, None] * rows[0][None, :] + rows[1][None, :]).double() * SCALE
    return M


def _hplai_matrix(n, seed, nrhs=1):
    """(O, d, B): O[j, i] = a_ij with a zero diagonal, the diagonal, nrhs right-hand sides as rows."""
    M = _lcg_matrix(n, seed, nrhs)
    O, B = M[:n], M[n:].clone()
    O.diagonal().zero_()
    d = torch.zeros(n, dtype=torch.float64, device=DEV)
    for j in range(0, n, 4096):
        d += O[j:j + 4096].abs().sum(0)
    return O, d, B


def _times(O, X):
    """X O for rows X, summed over chunks of O's rows."""
    Y = torch.zeros_like(X)
    for j in range(0, O.shape[0], 4096):
        Y += X[:, j:j + 4096] @ O[j:j + 4096]
    return Y


def _jacobi(mul, d, B, steps):
    """x = (b - O x) / d to its fixed point: the off-diagonal part is a small perturbation."""
    X = B / d
    for _ in range(steps):
        X = (B - mul(X)) / d
    return X


def exact(case, seed):
    f = case["form"]
    seed = int(seed)
    if f == "solve":
        O, d, B = _hplai_matrix(case["n"], seed)
        return dict(x=_jacobi(lambda X: _times(O, X), d, B, 24)[0], converged=None)
    if f == "autograd":
        A, B, W = _dense(case["n"], case["k"], seed)
        d = A.diagonal().clone()
        A.diagonal().zero_()
        At = A.t().contiguous()
        X = _jacobi(lambda Y: _times(At, Y), d, B.t().contiguous(), 24)       # rows of X^T
        Lam = _jacobi(lambda Y: _times(A, Y), d, W.t().contiguous(), 24)      # A^T Lambda = W
        return dict(X=X.t(), dA=-(Lam.t() @ X), dB=Lam.t())
    if f == "batch":
        xs = []
        for n, r, sd in zip(*_batch(case, seed)):
            if int(n) < 2:
                return None
            O, d, B = _hplai_matrix(int(n), int(sd), int(r))
            # below an order of about 40 the off-diagonal part is no small perturbation
            if n < 40:
                M = O.clone()
                M.diagonal().copy_(d)
                xs.append(torch.linalg.solve(M.t().cpu(), B.t().cpu()).t().reshape(-1))
            else:
                xs.append(_jacobi(lambda X: X @ O, d, B, 40).reshape(-1).cpu())
        return dict(x=torch.cat(xs), info=None)
    if f == "residual":
        n = case["n"]
        O, d, _ = _hplai_matrix(n, seed)
        rhs = _uniform((n,), _gen(seed), torch.float64)
        x = rhs / d
        return rhs - _times(O, x[None, :])[0] - d * x
    if f == "generate":
        O, d, B = _hplai_matrix(case["n"], seed)
        O.diagonal().copy_(d)
        return dict(A=O, d=d, b=B[0])
    if f == "panel":
        D, L, U = (t.double() for t in _panel(case, seed))
        b = case["b"]
        F = D.t().contiguous()
        for k in range(b - 1):
            F[k + 1:, k] /= F[k, k]
            F[k + 1:, k + 1:] -= F[k + 1:, k, None] * F[k, None, k + 1:]
        one = torch.tril(F, -1) + torch.eye(b, dtype=torch.float64, device=DEV)
        Lx = torch.linalg.solve_triangular(torch.triu(F), L.t(), upper=True, left=False)
        Ux = torch.linalg.solve_triangular(one, U.t(), upper=False, unitriangular=True)
        return dict(D=F.t(), L=Lx.t(), U=Ux.t(), info=None)
    if f == "update":
        m, n, b, fmt = case["m"], case["n"], case["b"], case["fmt"]
        L, U, C = _update(case, seed)
        Cx = C.double()
        for t in range(case["slices"]):
            Lt = _quantized(L[t * b:(t + 1) * b].t().contiguous(), b, fmt)
            Ut = _quantized(U[:, t * b:(t + 1) * b].contiguous(), b, fmt)
            Cx -= Ut @ Lt.t()
        return dict(C=Cx, Lq=None, Uq=None) if fmt == "f16" else dict(C=Cx, Lq=None, Uq=None, eL=None, eU=None)
    a, b, c = _seam(case, seed)
    return c.double() - b.double() @ a.double()


def _quantized(P, tb, fmt):
    """The rows of P rounded to the format with one power of two per tb rows, as FP64 values."""
    if fmt == "f16":
        return P.half().double()
    top, frac = (448.0, 1.75) if fmt == "e4m3" else (65504.0, 2.0 - 2.0 ** -10)
    out = torch.empty(P.shape, dtype=torch.float64, device=DEV)
    for i in range(0, P.shape[0], tb):
        R = P[i:i + tb].double()
        mant, ex = math.frexp(float(R.abs().max()))       # amax = 2 mant * 2^(ex - 1)
        e = (8 if fmt == "e4m3" else 15) - (ex - 1) - (1 if 2.0 * mant > frac else 0)
        S = (R * 2.0 ** e).float().clamp(-top, top)
        out[i:i + tb] = (S.to(torch.float8_e4m3fn) if fmt == "e4m3" else S.half()).double() * 2.0 ** -e
    return out
