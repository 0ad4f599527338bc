"""The doubling solver of left_polar_pullback! against the conjugate-gradient
path (maxiter = 47 keeps it) and the oracle's rule.

Both solve the same equation to relative residual 1e-14 or better; with
kappa(P) <= 30 here the solutions agree to 30 * 1e-14 and the rule's own
products add n u, so 1e-11 bounds the difference with a factor of ten."""
import numpy as np
import pytest
import torch

import mak_mi355x as mak
from oracle import mak_oracle as O

pytestmark = pytest.mark.gpu


def padded(x, dev, pad):
    """(batch, r, c) device tensor with leading dimension r + pad and a gap between matrices."""
    b, r, c = x.shape
    buf = torch.full((b, c + 1, r + pad), float("nan"), dtype=torch.from_numpy(x).dtype, device=dev)
    v = buf.transpose(1, 2)[:, :r, :c]
    v.copy_(torch.from_numpy(x).to(dev))
    return v


def run(dev, W, P, dW, dP, m, n, pad, maxiter):
    b = W.shape[0]
    dA = padded(np.ones((b, m, n), dtype=W.dtype), dev, pad)
    _, it = mak.left_polar_pullback_batched_(dA, padded(W, dev, pad), padded(P, dev, pad), padded(dW, dev, pad),
                                             None if dP is None else padded(dP, dev, pad), maxiter=maxiter)
    return dA.cpu().numpy(), it


# n at the edges of the 32-column steps and 64-column tiles
@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
@pytest.mark.parametrize("batch,m,n,pad", [(1, 3, 1, 0), (2, 9, 4, 1), (3, 40, 17, 0), (1, 70, 32, 2), (2, 100, 33, 0),
                                           (5, 130, 64, 3), (2, 200, 65, 0), (1, 300, 100, 0), (2, 400, 160, 1)])
def test_matches_cg_and_the_rule(batch, m, n, pad, dt, dev):
    A = [O.gaussian(m, n, dt, seed=7 * m + b) for b in range(batch)]
    W, P = (np.stack(x) for x in zip(*[O.left_polar_svd(a) for a in A]))
    dW = np.stack([O.gaussian(m, n, dt, seed=900 + b) for b in range(batch)])
    dP = np.stack([O.gaussian(n, n, dt, seed=950 + b) for b in range(batch)])
    for d2 in (dP, None):
        got, it = run(dev, W, P, dW, d2, m, n, pad, 200)
        cg, _ = run(dev, W, P, dW, d2, m, n, pad, 47)
        assert it <= 8
        assert np.linalg.norm(got - cg) < 1e-11 * np.linalg.norm(cg)
        for b in range(batch):
            ref = O.left_polar_pullback(np.ones((m, n), dtype=dt), A[b], (W[b], P[b]),
                                        (dW[b], None if d2 is None else d2[b]))
            assert np.linalg.norm(got[b] - ref) < 1e-11 * np.linalg.norm(ref)


@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
def test_a_batch_that_does_not_qualify_keeps_the_old_path(dt, dev):
    """One matrix with kappa(P) = 1e5 in the batch: the whole batch goes through
    CG / the eigendecomposition; an indefinite P is refused as before."""
    n = 40
    W = np.stack([np.linalg.qr(O.gaussian(n, n, dt, seed=b))[0] for b in range(2)])
    lam = np.stack([np.linspace(1, 2, n), np.logspace(0, -5, n)])
    P = np.stack([(W[1 - b] * lam[b]) @ W[1 - b].conj().T for b in range(2)])
    P = 0.5 * (P + P.conj().transpose(0, 2, 1))
    dW = np.stack([O.gaussian(n, n, dt, seed=20 + b) for b in range(2)])
    got, it = run(dev, W, P, dW, None, n, n, 0, 200)
    for b in range(2):
        ref = O.left_polar_pullback(np.ones((n, n), dtype=dt), None, (W[b], P[b]), (dW[b], None))
        assert np.linalg.norm(got[b] - ref) < 1e-9 * np.linalg.norm(ref)
    P[0] -= 1.5 * np.eye(n)
    with pytest.raises(mak.NumericalError):
        run(dev, W, P, dW, None, n, n, 0, 200)
