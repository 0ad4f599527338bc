"""The last two products of left_polar_pullback! in one launch (real data, n a
multiple of 16, batches with enough tiles) against the conjugate-gradient path
(maxiter = 47), whose products are separate, and the oracle's rule.

Both solve the Sylvester equation to relative residual 1e-14 or better; with
kappa(P) <= 30 the solutions agree to 30 * 1e-14 and the products add n u, so
1e-11 bounds the difference with a factor of ten."""
import numpy as np
import pytest
import torch

import mak_mi355x as mak
from oracle import mak_oracle as O

pytestmark = pytest.mark.gpu


def padded(x, dev, pad):
    b, r, c = x.shape
    buf = torch.full((b, c + 1, r + pad), float("nan"), dtype=torch.float64, device=dev)
    v = buf.transpose(1, 2)[:, :r, :c]
    v.copy_(torch.from_numpy(x).to(dev))
    return v


# one 16-column K-tile, ragged rows on 64 tiles, 128 tiles, unequal leading
# dimensions of the two left operands, and n that stays on two products
@pytest.mark.parametrize("batch,m,n,pads", [(130, 70, 16, (0, 0)), (40, 200, 64, (1, 1)), (60, 333, 80, (0, 0)),
                                            (40, 260, 160, (3, 3)), (40, 200, 64, (0, 2)), (40, 200, 60, (0, 0))])
def test_one_launch_matches_two(batch, m, n, pads, dev):
    A = [O.gaussian(m, n, np.float64, seed=5 * m + b) for b in range(batch)]
    W, P = (np.stack(x) for x in zip(*[O.left_polar_svd(a) for a in A]))
    dW = np.stack([O.gaussian(m, n, np.float64, seed=900 + b) for b in range(batch)])
    dP = np.stack([O.gaussian(n, n, np.float64, seed=950 + b) for b in range(batch)])
    outs = []
    for maxiter in (200, 47):
        dA = padded(np.ones((batch, m, n)), dev, pads[0])
        mak.left_polar_pullback_batched_(dA, padded(W, dev, pads[0]), padded(P, dev, 0), padded(dW, dev, pads[1]),
                                         padded(dP, dev, 0), maxiter=maxiter)
        outs.append(dA.cpu().numpy())
    assert np.linalg.norm(outs[0] - outs[1]) < 1e-11 * np.linalg.norm(outs[1])
    for b in (0, batch // 2, batch - 1):
        ref = O.left_polar_pullback(np.ones((m, n)), A[b], (W[b], P[b]), (dW[b], dP[b]))
        assert np.linalg.norm(outs[0][b] - ref) < 1e-11 * np.linalg.norm(ref)
