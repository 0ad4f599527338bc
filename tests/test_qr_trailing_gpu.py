"""The trailing columns of qr_full! and the signs of positive = false, formed
from the CholeskyQR2 factors (Householder reconstruction), against the
reflectors themselves.

The reference of a matrix A with positive-gauge QR factors Q R is built in
numpy: the LU of Q - [S; 0] without pivoting, s_j = -p_j / |p_j| of the j-th
pivot, gives the reflectors' V (its L) and T = -U S^H V_1^{-H}; the
Householder QR's Q is I - V T V^H and its R is S R.  Q and R themselves are
determined to about sqrt(n) u kappa(A), and M = Q_1 - S that the trailing
columns come from has pivots of magnitude 1 to 2 and a condition number of a
few times n, so the bounds are 1e-13 kappa(A) per column (u n^(3/2) at n = 300
is 6e-13 for an error of one sign throughout, and errors of random sign stay
some ten times below 1e-13)."""
import numpy as np
import pytest
import torch

import mak_mi355x as mak
from oracle import mak_oracle as O

pytestmark = pytest.mark.gpu


def householder_reference(A):
    m, n = A.shape
    Q, R = O.qr_compact(A)
    B = Q.astype(Q.dtype, copy=True)
    s = np.zeros(n, dtype=Q.dtype)
    for j in range(n):
        p = B[j, j]
        s[j] = -(p / abs(p)) if p != 0 else -1.0
        B[j, j] = p - s[j]
        B[j + 1:, j] /= B[j, j]
        B[j + 1:, j + 1:] -= np.outer(B[j + 1:, j], B[j, j + 1:])
    V = np.tril(B, -1)
    V[np.arange(n), np.arange(n)] = 1.0
    U = np.triu(B[:n])
    T = -(U * s.conj()[None, :]) @ np.linalg.inv(V[:n]).conj().T
    return Q, R, s, np.eye(m, dtype=Q.dtype) - V @ (T @ V.conj().T)


# one and several 32-column steps, a padded last step, partial 64-column tiles,
# one trailing column, and 64 rows or more below the last panel (complex data
# takes this path only then)
SHAPES = [(160, 64), (129, 65), (200, 96), (300, 127), (193, 128), (400, 130), (700, 300)]


@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
@pytest.mark.parametrize("m,n", SHAPES)
def test_full_q_is_the_product_of_the_reflectors(m, n, dt, dev):
    A = O.gaussian(m, n, dt, seed=3 * m + n)
    Q, R, s, H = householder_reference(A)
    tol = 1e-13 * max(1.0, np.linalg.cond(A))
    At = mak.colmajor(torch.from_numpy(np.asfortranarray(A)).to(dev))
    for positive in (True, False):
        alg = mak.MI355XHouseholder(positive=positive)
        Qf, Rf = (x.cpu().numpy() for x in mak.qr_full(At, alg))
        Qc, Rc = (x.cpu().numpy() for x in mak.qr_compact(At, alg))
        d = np.ones(n, dtype=dt) if positive else s
        assert np.linalg.norm(Qf[:, :n] - Q * d.conj()) < tol * np.sqrt(n)
        assert np.linalg.norm(Qf[:, n:] - H[:, n:]) < tol * np.sqrt(m)
        assert np.linalg.norm(Rf[:n] - d[:, None] * R) < tol * np.linalg.norm(R)
        assert np.all(Rf[n:] == 0) and np.all(np.tril(Rf, -1) == 0)
        assert np.array_equal(Qc, Qf[:, :n]) and np.array_equal(Rc, Rf[:n])
        assert np.linalg.norm(Qf.conj().T @ Qf - np.eye(m)) < 1e-12


@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
def test_full_q_one_trailing_column_and_padded_ld(dt, dev):
    """m = n + 1 (complex data: m = n + 64, its smallest), and outputs with
    leading dimensions beyond their rows: nothing outside them is written."""
    n = 100
    m = n + (64 if dt == np.complex128 else 1)
    A = O.gaussian(m, n, dt, seed=8)
    _, R, _, H = householder_reference(A)
    tol = 1e-13 * max(1.0, np.linalg.cond(A))
    At = mak.colmajor(torch.from_numpy(np.asfortranarray(A)).to(dev))
    Qp = torch.full((m, m + 3), 7.0, dtype=At.dtype, device=dev).t()
    Rp = torch.full((n, m + 5), 7.0, dtype=At.dtype, device=dev).t()
    mak.qr_full_(At, (Qp[:m], Rp[:m]))
    assert np.linalg.norm(Qp[:m, n:].cpu().numpy() - H[:, n:]) < tol * np.sqrt(m)
    assert np.linalg.norm(Rp[:n].cpu().numpy() - R) < tol * np.linalg.norm(R)
    assert torch.all(Rp[n:m] == 0) and torch.all(Qp[m:] == 7) and torch.all(Rp[m:] == 7)


@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
def test_full_q_of_a_rejected_input(dt, dev):
    """A rank-deficient input is rejected on the device: the gated launches
    leave the outputs to the Householder path."""
    A = O.gaussian(260, 80, dt, seed=5)
    A[:, 40] = A[:, 7]
    At = mak.colmajor(torch.from_numpy(np.asfortranarray(A)).to(dev))
    for positive in (True, False):
        Q, R = (x.cpu().numpy() for x in mak.qr_full(At, mak.MI355XHouseholder(positive=positive)))
        assert np.linalg.norm(Q @ R - A) < 1e-13 * np.linalg.norm(A)
        assert np.linalg.norm(Q.conj().T @ Q - np.eye(260)) < 1e-12
        assert np.all(np.tril(R, -1) == 0)
