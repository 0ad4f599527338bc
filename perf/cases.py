"""The workloads that speed is measured on: the factorizations and reverse rules
of this package as a tensor-network or numerical program calls them.

``listed()`` names twelve cases over the whole range, ``draw(rng)`` gives more
of the same ranges, ``prepare`` makes what a program holds before the call,
``run`` is one pass through the public entry points, ``work`` the bytes and
flops that the task cannot do without, and ``exact`` the same outputs from
plain LAPACK / torch in 64 bits.

Kinds of case (Float64 unless ``complex``):

* ``qr_compact``, ``qr_full``, ``lq_compact``: one matrix, the positive gauge
  (the default) or, for drawn compact QRs, also without it; the input is kept
  (the out-of-place entry point copies it, as the reference's ``copy_input``).
* ``left_polar``, ``right_polar``: one matrix with singular values spaced
  evenly in their logarithm from 1 down to 1 / ``cond``, or Gaussian (``cond``
  0).  ``precision`` 32 is the reduced-precision bulk; a program that asks for
  it keeps its factors in 32 bits.
* ``batched_qr``: the blocks of a block-sparse tensor, m log-uniform in
  [16, mmax] and n uniform in [8, m], in one flat buffer: the program keeps a
  plan, writes the next tensor's blocks into the buffer and executes the plan.
* ``qr_pullback``, ``left_polar_pullback``: the reverse rule of a batch of tall
  Gaussian matrices from the tape (QR) or the factors (polar) that the forward
  pass left, onto a zero gradient.
"""
import math
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT / "matrixalgebrakit.jl_amd") not in sys.path:
    sys.path.insert(0, str(ROOT / "matrixalgebrakit.jl_amd"))

import mak_mi355x as mak  # noqa: E402

DEV = "cuda:0"


def listed():
    return [
        # a single small tensor block: launches, synchronisation and host work
        {"name": "qr_compact_57x33", "kind": "qr_compact", "m": 57, "n": 33, "complex": False, "positive": True},
        # one dense matrix of ordinary size
        {"name": "qr_compact_1024x512", "kind": "qr_compact", "m": 1024, "n": 512, "complex": False,
         "positive": True},
        # the tall matrix of the benchmark's headline
        {"name": "qr_compact_8192x1024", "kind": "qr_compact", "m": 8192, "n": 1024, "complex": False,
         "positive": True},
        # a wide complex matrix of odd size: the right orthogonalization of a sweep
        {"name": "lq_compact_c64_777x3001", "kind": "lq_compact", "m": 777, "n": 3001, "complex": True},
        # the full square factor of the tall matrix
        {"name": "qr_full_8192x1024", "kind": "qr_full", "m": 8192, "n": 1024, "complex": False},
        # the benchmark's polar decomposition, in FP64
        {"name": "left_polar_4096", "kind": "left_polar", "m": 4096, "n": 4096, "complex": False, "cond": 0.0,
         "precision": 64},
        # the same size with the reduced-precision bulk, on an ill-conditioned matrix
        {"name": "left_polar_4096_p32", "kind": "left_polar", "m": 4096, "n": 4096, "complex": False,
         "cond": 1e4, "precision": 32},
        # a wide complex matrix of odd size: a canonical form from the right
        {"name": "right_polar_c64_501x1203", "kind": "right_polar", "m": 501, "n": 1203, "complex": True,
         "cond": 0.0, "precision": 64},
        # thousands of uneven blocks in one call
        {"name": "batched_qr_4096", "kind": "batched_qr", "count": 4096, "mmax": 1024, "complex": False},
        # the same in complex arithmetic
        {"name": "batched_qr_c64_1024", "kind": "batched_qr", "count": 1024, "mmax": 1024, "complex": True},
        # the reverse rules on the benchmark's batch of tall matrices
        {"name": "qr_pullback_256x2048x256", "kind": "qr_pullback", "batch": 256, "m": 2048, "n": 256,
         "complex": False},
        {"name": "left_polar_pullback_256x2048x256", "kind": "left_polar_pullback", "batch": 256, "m": 2048,
         "n": 256, "complex": False},
    ]


def _log_int(rng, lo, hi):
    """An integer spread evenly over [lo, hi] in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["qr_compact", "qr_compact", "lq_compact", "qr_full", "left_polar", "left_polar",
                       "right_polar", "batched_qr", "batched_qr", "qr_pullback", "left_polar_pullback"])
    cplx = rng.random() < 0.4
    if kind == "qr_compact":
        m = _log_int(rng, 16, 8192)
        return {"kind": kind, "m": m, "n": _log_int(rng, 8, min(m, 1024)), "complex": cplx,
                "positive": rng.random() < 0.75}
    if kind == "lq_compact":
        n = _log_int(rng, 16, 8192)
        return {"kind": kind, "m": _log_int(rng, 8, min(n, 1024)), "n": n, "complex": cplx}
    if kind == "qr_full":
        m = _log_int(rng, 64, 4096 if cplx else 8192)
        return {"kind": kind, "m": m, "n": _log_int(rng, 16, min(m, 1024)), "complex": cplx}
    if kind in ("left_polar", "right_polar"):
        low = kind == "left_polar" and not cplx and rng.random() < 0.4
        n = _log_int(rng, 256 if low else 32, 2048 if cplx else 4096)
        m = min(4096, int(n * rng.uniform(1.0, 3.0)))
        if kind == "right_polar":
            m, n = n, m
        return {"kind": kind, "m": m, "n": n, "complex": cplx, "cond": float("%.3g" % 10.0 ** rng.uniform(1.0, 4.0)),
                "precision": 32 if low else 64}
    if kind == "batched_qr":
        return {"kind": kind, "count": _log_int(rng, 64, 1024 if cplx else 4096), "mmax": _log_int(rng, 128, 1024),
                "complex": cplx}
    n = _log_int(rng, 16, 256)
    return {"kind": kind, "batch": _log_int(rng, 1, 64 if cplx else 256), "m": int(n * rng.uniform(2.0, 8.0)), "n": n,
            "complex": cplx}


# ---------------------------------------------------------------------------
# inputs, from the case and the seed alone
# ---------------------------------------------------------------------------
def _dtype(case):
    return torch.complex128 if case["complex"] else torch.float64


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _gauss(g, dtype, *shape):
    return torch.randn(shape, generator=g, dtype=dtype, device=DEV)


def _matrix(g, dtype, m, n):
    """A column-major Gaussian m x n matrix."""
    return _gauss(g, dtype, n, m).t()


def _polar_input(case, seed):
    g, dt, m, n = _generator(seed), _dtype(case), case["m"], case["n"]
    if not case["cond"]:
        return _matrix(g, dt, m, n)
    k = min(m, n)
    U, V = torch.linalg.qr(_gauss(g, dt, m, k))[0], torch.linalg.qr(_gauss(g, dt, n, k))[0]
    s = torch.logspace(0, -math.log10(case["cond"]), k, dtype=torch.float64, device=DEV)
    return mak.colmajor((U * s) @ V.mH)


def _shapes(case, seed):
    return mak.block_shapes(case["count"], seed=seed, mmax=case["mmax"])


def _views(flat, shapes, size):
    out, at = [], 0
    for m, n in shapes:
        r, c = size(m, n)
        out.append(flat[at:at + r * c].view(c, r).t())
        at += r * c
    return out


def _cotangent(g, dt, b, r, c):
    return _gauss(g, dt, b, c, r).transpose(1, 2)


def _batch(case, seed):
    """The matrices A_b and the cotangents of the reverse rules."""
    g, dt, b, m, n = _generator(seed), _dtype(case), case["batch"], case["m"], case["n"]
    A = _cotangent(g, dt, b, m, n)
    d1, d2 = _cotangent(g, dt, b, m, n), _cotangent(g, dt, b, n, n)
    if case["kind"] == "qr_pullback":
        d2 = mak.colmajor_batch(torch.triu(d2))
    return A, d1, d2


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind in ("qr_compact", "qr_full", "lq_compact"):
        s["A"] = _matrix(_generator(seed), _dtype(case), case["m"], case["n"])
        s["alg"] = mak.MI355XHouseholder(positive=case.get("positive", True))
    elif kind in ("left_polar", "right_polar"):
        s["A"] = _polar_input(case, seed)
        s["alg"] = mak.MI355XPolar(precision=case["precision"])
    elif kind == "batched_qr":
        # the block structure belongs to the network, the values to the seed
        shapes, dt, g = _shapes(case, 0), _dtype(case), _generator(seed)
        total = sum(m * n for m, n in shapes)
        s["next"] = _gauss(g, dt, total)
        s["blocks"] = torch.zeros(total, dtype=dt, device=DEV)
        s["Q"] = torch.zeros(total, dtype=dt, device=DEV)
        s["R"] = torch.zeros(sum(n * n for _, n in shapes), dtype=dt, device=DEV)
        s["plan"] = mak.BatchedQRPlan(_views(s["blocks"], shapes, lambda m, n: (m, n)),
                                      _views(s["Q"], shapes, lambda m, n: (m, n)),
                                      _views(s["R"], shapes, lambda m, n: (n, n)))
    elif kind == "qr_pullback":
        A, s["dQ"], s["dR"] = _batch(case, seed)
        fwd = [mak.qr_compact_rrule(a) for a in A]
        s["Awy"] = mak.colmajor_batch(torch.stack([t.Awy for _, _, t in fwd]))
        s["T"] = torch.stack([t.T for _, _, t in fwd])
        s["R"] = mak.colmajor_batch(torch.stack([r for _, r, _ in fwd]))
    else:
        A, s["dW"], s["dP"] = _batch(case, seed)
        fwd = [mak.left_polar(a) for a in A]
        s["W"] = mak.colmajor_batch(torch.stack([w for w, _ in fwd]))
        s["P"] = mak.colmajor_batch(torch.stack([p for _, p in fwd]))
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "qr_compact":
        return mak.qr_compact(s["A"], s["alg"])
    if kind == "qr_full":
        return mak.qr_full(s["A"], s["alg"])
    if kind == "lq_compact":
        return mak.lq_compact(s["A"], s["alg"])
    if kind in ("left_polar", "right_polar"):
        x, y = (mak.left_polar if kind == "left_polar" else mak.right_polar)(s["A"], s["alg"])
        return (x, y) if case["precision"] == 64 else (x.to(torch.float32), y.to(torch.float32))
    if kind == "batched_qr":
        s["blocks"].copy_(s["next"])
        s["plan"].execute()
        return s["Q"], s["R"]
    b, m, n = case["batch"], case["m"], case["n"]
    dA = mak.empty_colmajor_batch(b, m, n, _dtype(case), DEV).zero_()
    if kind == "qr_pullback":
        return mak.qr_pullback_batched_(dA, s["Awy"], s["T"], s["R"], s["dQ"], s["dR"])
    return mak.left_polar_pullback_batched_(dA, s["W"], s["P"], s["dW"], s["dP"])[0]


# ---------------------------------------------------------------------------
# the least work
# ---------------------------------------------------------------------------
def _qr_flops(m, n):
    """LAPACK's count of xGEQRF and xORGQR (compact factors)."""
    k = min(m, n)
    f = 2 * m * n * n - 2 * n ** 3 / 3 if m >= n else 2 * n * m * m - 2 * m ** 3 / 3
    return f + 4 * m * k * k - 2 * (m + k) * k * k + 4 * k ** 3 / 3


def work(case):
    es, fl = (16, 4) if case["complex"] else (8, 1)
    kind = case["kind"]
    if kind == "batched_qr":
        shapes = _shapes(case, 0)
        return {"bytes": es * sum(2 * m * n + n * n for m, n in shapes),
                "flops": fl * sum(_qr_flops(m, n) for m, n in shapes)}
    m, n = case["m"], case["n"]
    k = min(m, n)
    if kind in ("qr_compact", "lq_compact"):
        # at least as tall as wide once transposed
        return {"bytes": es * (m * n + k * (m + n)), "flops": fl * _qr_flops(max(m, n), k)}
    if kind == "qr_full":
        # the factorization, W = V T and Q = I - W V^H
        return {"bytes": es * (2 * m * n + m * m),
                "flops": fl * (3 * m * n * n - 2 * n ** 3 / 3 + 2 * m * m * n)}
    if kind in ("left_polar", "right_polar"):
        # QDWH from l0 = 1e-10: two QR-form and three Cholesky-form steps, then P
        h = max(m, n)
        qr = 4 * (h + k) * k * k - 4 * k ** 3 / 3 + 2 * h * k * k
        chol = 3 * h * k * k + k ** 3 / 3
        return {"bytes": es * (2 * m * n + k * k), "flops": fl * (2 * qr + 3 * chol + h * k * k)}
    b = case["batch"]
    if kind == "qr_pullback":
        # Q from the tape, dQ^H Q, R dR^H, Q X and the triangular solve
        return {"bytes": es * b * (3 * m * n + 2 * n * n), "flops": fl * b * (7 * m * n * n + n ** 3 / 3)}
    # W^H dW, the Sylvester equation through the eigenvectors of P, W C and dW P^-1
    return {"bytes": es * b * (3 * m * n + 2 * n * n), "flops": fl * b * (6 * m * n * n + 10 * n ** 3)}


# ---------------------------------------------------------------------------
# the outputs from plain LAPACK / torch in 64 bits
# ---------------------------------------------------------------------------
def _gauge(Q, R):
    """The positive gauge: R's diagonal real and non-negative."""
    k = min(R.shape)
    d = torch.diagonal(R)
    ph = torch.where(d == 0, torch.ones_like(d), d / d.abs().clamp_min(1e-300))
    Q = Q.clone()
    Q[:, :k] *= ph
    R = R.clone()
    R[:k] *= ph.conj()[:, None]
    return Q, R


def _unitary_polar(A):
    """(U, H) of the square A = U H by Newton's iteration with Frobenius scaling."""
    X = A
    for _ in range(40):
        Y = torch.linalg.inv(X).mH
        z = torch.sqrt(torch.linalg.matrix_norm(Y) / torch.linalg.matrix_norm(X))
        new = 0.5 * (z * X + Y / z)
        done = torch.linalg.matrix_norm(new - X) <= 1e-8 * torch.linalg.matrix_norm(new)
        X = new
        if bool(done):
            break
    Y = torch.linalg.inv(X).mH
    X = 0.5 * (X + Y)
    H = X.mH @ A
    return X, 0.5 * (H + H.mH)


def _left_polar(A):
    m, n = A.shape
    if m == n:
        return _unitary_polar(A)
    Q, R = torch.linalg.qr(A.cpu())
    U, H = _unitary_polar(R.to(A.device))
    return Q.to(A.device) @ U, H


def exact(case, seed):
    kind = case["kind"]
    if kind in ("qr_compact", "qr_full", "lq_compact"):
        A = _matrix(_generator(seed), _dtype(case), case["m"], case["n"]).cpu()
        if kind == "lq_compact":
            Q, R = _gauge(*torch.linalg.qr(A.mH))
            return R.mH.resolve_conj(), Q.mH.resolve_conj()
        Q, R = torch.linalg.qr(A, mode="complete" if kind == "qr_full" else "reduced")
        return _gauge(Q, R) if case.get("positive", True) else (Q, R)
    if kind in ("left_polar", "right_polar"):
        A = _polar_input(case, seed)
        if kind == "left_polar":
            W, P = _left_polar(A)
            return W, P
        W, P = _left_polar(A.mH)
        return P, W.mH.resolve_conj()
    if kind == "batched_qr":
        shapes, dt = _shapes(case, 0), _dtype(case)
        flat = _gauss(_generator(seed), dt, sum(m * n for m, n in shapes)).cpu()
        Qf, Rf = torch.zeros_like(flat), torch.zeros(sum(n * n for _, n in shapes), dtype=dt)
        for A, Qv, Rv in zip(_views(flat, shapes, lambda m, n: (m, n)), _views(Qf, shapes, lambda m, n: (m, n)),
                             _views(Rf, shapes, lambda m, n: (n, n))):
            Q, R = _gauge(*torch.linalg.qr(A))
            Qv.copy_(Q)
            Rv.copy_(R)
        return Qf, Rf
    A, d1, d2 = _batch(case, seed)
    dA = torch.empty_like(A)
    for b in range(case["batch"]):
        a, x, y = A[b].cpu(), d1[b].cpu(), d2[b].cpu()
        if kind == "qr_pullback":
            # dA = (dQ + Q (tril(M) + tril(M, -1)^H)) R^-H, M = R dR^H - dQ^H Q
            # (a real diagonal: only the gauge's freedom is left out)
            Q, R = _gauge(*torch.linalg.qr(a))
            M = R @ y.mH - x.mH @ Q
            L = torch.tril(M, -1)
            D = torch.diag(torch.diagonal(M).real).to(M.dtype)
            dA[b] = torch.linalg.solve_triangular(R.mH, x + Q @ (L + L.mH + D), upper=False, left=False).to(DEV)
        else:
            # dA = W (C + dP) + (1 - W W^H) dW P^-1 with P C + C P = M - M^H, M = W^H dW - dP P
            U, s, Vh = torch.linalg.svd(a, full_matrices=False)
            W, P = U @ Vh, (Vh.mH * s.to(Vh.dtype)) @ Vh
            y = 0.5 * (y + y.mH)
            M = W.mH @ x - y @ P
            K = Vh @ (M - M.mH) @ Vh.mH / (s[:, None] + s[None, :])
            C = Vh.mH @ K @ Vh + y
            Z = ((x @ Vh.mH) / s.to(Vh.dtype)) @ Vh
            dA[b] = (W @ C + Z - W @ (W.mH @ Z)).to(DEV)
    return dA
