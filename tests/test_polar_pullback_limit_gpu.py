"""left_polar_pullback! near the limits of its doubling solver: it finishes every
batch that it takes, in as many steps as its recursion on P's eigenvalues takes,
and a batch just beyond goes to conjugate gradients or the eigendecomposition.

The equation P C + C P = F has condition number kappa(P), and so has P^{-1}: both
the solvers and the oracle are within a few n u kappa(P), the bound here (8 n u
kappa relative, 1e-9 at n = 512, kappa = 7e3)."""
import numpy as np
import pytest
import torch

import mak_mi355x as mak
from oracle import mak_oracle as O

pytestmark = pytest.mark.gpu


def steps(lam):
    """Steps of M <- M^2 until |M^(2^(K-1))|_F^4 <= 1e-17."""
    s = lam.mean()
    M2, k = ((lam - s) / (lam + s)) ** 2, 0
    while True:
        k += 1
        if M2.sum() ** 2 <= 1e-17:
            return k
        M2 = M2 ** 2


def one_small(n, c):
    lam = np.ones(n)
    lam[-1] = 1.0 / (c * n)
    return lam


def small_and_large(n, small, large):
    lam = np.ones(n)
    lam[0], lam[-1] = large, small
    return lam


CASES = [(256, one_small(256, 14.0), True), (512, one_small(512, 14.0), True), (64, one_small(64, 17.0), False),
         (300, small_and_large(300, 1.0 / 900, 300.0), True), (300, small_and_large(300, 1.0 / 3000, 300.0), False),
         (130, np.linspace(0.07, 1.0, 130), True), (1100, one_small(1100, 14.5), False)]


@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
@pytest.mark.parametrize("n,lam,taken", CASES)
def test_at_the_limit(n, lam, taken, dt, dev):
    m = n + 5
    q = lam.mean() * (1.0 / lam).mean()
    assert (q <= min(16.0, 16384.0 / n)) == taken
    W = np.linalg.qr(O.gaussian(m, n, dt, seed=n))[0]
    V = np.linalg.qr(O.gaussian(n, n, dt, seed=n + 1))[0]
    P = (V * lam) @ V.conj().T
    P = 0.5 * (P + P.conj().T)
    dW, dP = O.gaussian(m, n, dt, seed=n + 2), O.gaussian(n, n, dt, seed=n + 3)

    def up(x):
        return mak.colmajor_batch(torch.from_numpy(np.ascontiguousarray(x))[None].to(dev))

    dA = mak.empty_colmajor_batch(1, m, n, torch.from_numpy(W).dtype, dev).zero_()
    _, it = mak.left_polar_pullback_batched_(dA, up(W), up(P), up(dW), up(dP))
    if taken:
        assert it == steps(lam) <= 18
    # C in P's eigenvectors
    K = W.conj().T @ dW
    H = 0.5 * (dP + dP.conj().T)
    M = K - H @ P
    F = V.conj().T @ (M - M.conj().T) @ V
    C = V @ (F / (lam[:, None] + lam[None, :])) @ V.conj().T
    ref = W @ (C + H) + (dW - W @ K) @ ((V / lam) @ V.conj().T)
    got = dA[0].cpu().numpy()
    assert np.linalg.norm(got - ref) <= 8 * n * 2.0 ** -53 * (lam.max() / lam.min()) * np.linalg.norm(ref)
