"""||A - Q R|| of inputs with two nearly parallel columns, on every CholeskyQR2
route that forms Q1 with a computed inverse.

The residual of A X, X a computed inverse of R1, is about u cond(R1); substitution
with a step of refinement leaves a few u.  The condition numbers here are ones
that each route accepts.  Bound: 1e-14 (90 u) relative to ||A||, as the other
tests of these paths ask of their well-conditioned inputs: Householder QR is
within a few sqrt(n) u of it.
"""
import numpy as np
import pytest
import torch

import mak_mi355x as mak
from oracle import mak_oracle as O

pytestmark = pytest.mark.gpu
DTYPES = pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])


def near_parallel(m, n, j, cond, dt, seed):
    """Gaussian, but for column j at a distance of about 1 / cond from column 0."""
    A = O.gaussian(m, n, dt, seed=seed)
    A[:, j] = A[:, 0] + A[:, j] / cond
    return A


def to_dev(A, dev):
    return mak.colmajor(torch.from_numpy(np.asfortranarray(A)).to(dev))


def check(A, Q, R):
    k = min(A.shape)
    Q, R = Q.cpu().numpy(), R.cpu().numpy()
    res = np.linalg.norm(A - Q[:, :k] @ R[:k]) / np.linalg.norm(A)
    orth = np.linalg.norm(Q.conj().T @ Q - np.eye(Q.shape[1])) / np.sqrt(Q.shape[1])
    assert res <= 1e-14 and orth <= 1e-14, (res, orth)


@DTYPES
@pytest.mark.parametrize("m,n,j", [(57, 33, 1), (57, 40, 1), (63, 63, 31), (40, 32, 31), (60, 45, 44), (63, 64 - 1, 62)])
def test_small_near_parallel(m, n, j, dt, dev):
    for cond in (1e2, 1e3):
        A = near_parallel(m, n, j, cond, dt, 3)
        check(A, *mak.qr_compact(to_dev(A, dev)))


@DTYPES
@pytest.mark.parametrize("m,n,j", [(64, 33, 32), (100, 63, 32), (600, 40, 1), (600, 40, 39), (5000, 63, 62), (700, 32, 1)])
def test_tall_near_parallel(m, n, j, dt, dev):
    for cond in (1e2, 1e4):
        A = near_parallel(m, n, j, cond, dt, 5)
        check(A, *mak.qr_compact(to_dev(A, dev)))


@DTYPES
def test_whole_blocks_near_parallel(dt, dev):
    """Columns of one 64-column tile and of different ones; one pass and two."""
    host = [near_parallel(m, n, j, cond, dt, 7)
            for m, n, j in ((64, 40, 1), (100, 64, 32), (130, 128, 127), (200, 150, 140), (300, 190, 65), (400, 64, 63))
            for cond in (1e2, 1e3, 1e5)]
    plan = mak.BatchedQRPlan([to_dev(h, dev) for h in host])
    Qs, Rs = plan.execute()
    torch.cuda.synchronize()
    for h, q, r in zip(host, Qs, Rs):
        check(h, q, r)
    plan.close()


@DTYPES
@pytest.mark.parametrize("full,positive", [(True, True), (True, False), (False, False)])
@pytest.mark.parametrize("m,n,j", [(200, 64, 1), (200, 64, 33), (600, 160, 130), (700, 300, 299)])
def test_signed_and_full_near_parallel(m, n, j, full, positive, dt, dev):
    for cond in (1e2, 1e4):
        A = near_parallel(m, n, j, cond, dt, 9)
        f = mak.qr_full if full else mak.qr_compact
        check(A, *f(to_dev(A, dev), mak.MI355XHouseholder(positive=positive)))
