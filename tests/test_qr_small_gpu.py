"""qr_compact! of matrices with n <= m < 64 (one workgroup: CholeskyQR2 in LDS,
Householder QR in the same kernel when it is rejected) against the oracle.

Bounds: backward error and loss of orthogonality of QR on at most 63 rows are a
few u; 1e-14 (45 u) relative holds whatever the condition number.  Forward
errors of Q and R are a few condition numbers times u: 1e-12 to condition 1e3.
"""
import numpy as np
import pytest
import torch

import mak_mi355x as mak
from oracle import mak_oracle as O

pytestmark = pytest.mark.gpu

# edges of the 16-row waves, the 32-column blocks and the 4-row stages
SHAPES = [(1, 1), (3, 1), (5, 4), (16, 16), (17, 15), (31, 31), (32, 32), (33, 32), (33, 33), (47, 34), (57, 33),
          (63, 17), (63, 32), (63, 48), (63, 49), (63, 62), (63, 63)]


def conditioned(m, n, dt, cond, seed):
    rng = np.random.default_rng(seed)

    def ortho(r, c):
        x = rng.standard_normal((r, c))
        if dt == np.complex128:
            x = x + 1j * rng.standard_normal((r, c))
        return np.linalg.qr(x)[0]

    return (ortho(m, n) * np.logspace(0, -np.log10(cond), n)) @ ortho(n, n).conj().T


def factor(A, dev, with_r=True, pad=0):
    """Through mak.qr_compact_ on views with `pad` rows below each matrix."""
    m, n = A.shape
    dt = torch.complex128 if np.iscomplexobj(A) else torch.float64
    buf = [torch.full((n, r + pad), 7.0, dtype=dt, device=dev).t() for r in (m, m, n)]
    a, q, r = buf[0][:m], buf[1][:m], buf[2][:n]
    a.copy_(torch.from_numpy(A).to(dev))
    mak.qr_compact_(a, (q, r if with_r else torch.empty((0, 0), dtype=dt, device=dev)))
    torch.cuda.synchronize()
    for x, rows in ((buf[1], m), (buf[2], n)):
        assert (x[rows:] == 7.0).all()
    if not with_r:
        assert (buf[2] == 7.0).all()
    return q.cpu().numpy(), r.cpu().numpy()


def check(A, Q, R):
    assert np.all(np.isfinite(Q)) and np.all(np.isfinite(R))
    assert np.linalg.norm(A - Q @ R) <= 1e-14 * np.linalg.norm(A)
    assert np.linalg.norm(Q.conj().T @ Q - np.eye(Q.shape[1])) <= 1e-14 * np.sqrt(Q.shape[1])
    d = np.diagonal(R)
    assert np.all(d.real >= 0) and np.all(d.imag == 0) and np.array_equal(R, np.triu(R))


@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
@pytest.mark.parametrize("m,n", SHAPES)
def test_small_shapes(m, n, dt, dev):
    for cond, pad in ((10.0, 0), (1e3, 5)):
        A = conditioned(m, n, dt, cond, 100 * m + n)
        Q, R = factor(A, dev, pad=pad)
        check(A, Q, R)
        Qo, Ro = O.qr_compact(A)
        assert np.linalg.norm(Q - Qo) <= 1e-12 * np.linalg.norm(Qo)
        assert np.linalg.norm(R - Ro) <= 1e-12 * np.linalg.norm(Ro)
        assert np.array_equal(factor(A, dev, with_r=False)[0], Q)


@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
def test_small_rejected(dt, dev):
    """Inputs on both sides of the check, and rank-deficient ones, whose factors
    are the oracle's Householder factors where they are determined."""
    for m, n in ((40, 20), (60, 45), (63, 63)):
        for cond in (1e4, 1e5, 1e7, 1e10, 1e14):
            A = conditioned(m, n, dt, cond, m)
            check(A, *factor(A, dev, pad=1))
        Z = conditioned(m, n, dt, 10.0, m + 1)
        Z[:, 3] = 0.0
        D = conditioned(m, n, dt, 10.0, m + 2)
        D[:, n - 1] = D[:, 0]
        for A in (Z, D, np.zeros((m, n), dtype=dt), np.eye(m, n, dtype=dt)):
            Q, R = factor(A, dev)
            if np.any(A):
                check(A, Q, R)
            else:
                assert np.array_equal(Q, np.eye(m, n)) and not np.any(R)


def test_small_in_a_graph(dev):
    """One launch, no host check: a captured call replays on other values."""
    A = torch.zeros((33, 57), dtype=torch.float64, device=dev).t()
    Q, R = mak.initialize_output_qr(A, False)
    vals = [conditioned(57, 33, np.float64, c, 3) for c in (10.0, 1e9, 1e2)]
    mak.qr_compact_(A, (Q, R))
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        mak.qr_compact_(A, (Q, R))
    for v in vals:
        A.copy_(torch.from_numpy(v).to(dev))
        g.replay()
        torch.cuda.synchronize()
        got = (Q.cpu().numpy(), R.cpu().numpy())
        check(v, *got)
        A.copy_(torch.from_numpy(v).to(dev))
        e = mak.qr_compact(A)
        assert np.array_equal(got[0], e[0].cpu().numpy()) and np.array_equal(got[1], e[1].cpu().numpy())
