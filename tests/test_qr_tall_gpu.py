"""qr_compact! of matrices with m >= 64 rows and n < 64 columns (CholeskyQR2 in
three launches, the panels for a rejected input) against the oracle.

Bounds: backward error and loss of orthogonality stay at a few sqrt(n) u
whatever the condition number (1e-14 relative, 45 u); forward errors of Q and R
are a few condition numbers times u, 1e-12 to condition 1e3.
"""
import numpy as np
import pytest
import torch

import mak_mi355x as mak
from oracle import mak_oracle as O

pytestmark = pytest.mark.gpu

# edges of the 64-row strips, of the row ranges per workgroup (64 workgroups at
# most) and of the 32-column blocks
SHAPES = [(64, 1), (64, 63), (65, 33), (127, 32), (128, 31), (200, 20), (1000, 48), (4096, 33), (4097, 63), (9001, 8), (16384, 17), (16385, 17)]


def conditioned(m, n, dt, cond, seed):
    rng = np.random.default_rng(seed)

    def ortho(r, c):
        x = rng.standard_normal((r, c))
        if dt == np.complex128:
            x = x + 1j * rng.standard_normal((r, c))
        return np.linalg.qr(x)[0]

    return (ortho(m, n) * np.logspace(0, -np.log10(cond), n)) @ ortho(n, n).conj().T


def factor(A, dev, with_r=True, pad=0):
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
def test_tall_shapes(m, n, dt, dev):
    for cond, pad in ((10.0, 0), (1e3, 5)):
        A = conditioned(m, n, dt, cond, m + n)
        Q, R = factor(A, dev, pad=pad)
        check(A, Q, R)
        Qo, Ro = O.qr_compact(A)
        assert np.linalg.norm(Q - Qo) <= 1e-12 * np.linalg.norm(Qo)
        assert np.linalg.norm(R - Ro) <= 1e-12 * np.linalg.norm(Ro)
        assert np.array_equal(factor(A, dev, with_r=False)[0], Q)


@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
def test_tall_conditioning(dt, dev):
    """First- and second-order corrections, and inputs left to the panels."""
    for m, n in ((70, 20), (300, 45), (3000, 63)):
        for cond in (1e2, 3e3, 1e4, 3e4, 1e5, 1e6, 1e8, 1e12):
            A = conditioned(m, n, dt, cond, m)
            check(A, *factor(A, dev, pad=1))
        Z = conditioned(m, n, dt, 10.0, m + 1)
        Z[:, 3] = 0.0
        check(Z, *factor(Z, dev))
