"""Batched qr_compact! of whole blocks by CholeskyQR2 (64 x 64 tiles) against the
oracle and by its own properties.

Bounds: Householder QR of an m x n block has backward error and loss of
orthogonality of a few sqrt(n) u in practice; 1e-14 (45 u) is what the panel
schedule is held to, so the residual relative to ||A|| and
||Q^H Q - I|| / sqrt(n) must stay below it whatever the condition number.  Q and
R themselves are compared with the oracle where the condition number is at most
1e3: their forward error is a few condition numbers times u, below 1e-12.
"""
import numpy as np
import pytest
import torch

import mak_mi355x as mak
from oracle import mak_oracle as O

pytestmark = pytest.mark.gpu

# edges of the 64-row strips, 64-column tiles and 16- (8-) index stages, one to
# several block columns, the smallest blocks taken whole and their neighbours
EDGE = [(64, 1), (64, 8), (63, 20), (64, 40), (65, 17), (80, 63), (96, 64), (130, 65), (127, 66), (200, 128),
        (193, 129), (300, 190), (257, 192), (400, 257), (500, 320), (1000, 31), (1024, 449)]


def conditioned(m, n, dt, cond, seed):
    """m x n with singular values log-spaced from 1 to 1 / cond."""
    rng = np.random.default_rng(seed)

    def ortho(r, c):
        x = rng.standard_normal((r, c))
        if dt == np.complex128:
            x = x + 1j * rng.standard_normal((r, c))
        return np.linalg.qr(x)[0]

    return (ortho(m, n) * np.logspace(0, -np.log10(cond), n)) @ ortho(n, n).conj().T


def check(A, Q, R, forward):
    k = Q.shape[1]
    assert np.all(np.isfinite(Q)) and np.all(np.isfinite(R))
    assert np.linalg.norm(A - Q @ R) <= 1e-14 * np.linalg.norm(A), A.shape
    assert np.linalg.norm(Q.conj().T @ Q - np.eye(k)) <= 1e-14 * np.sqrt(k), A.shape
    d = np.diagonal(R)
    assert np.all(d.real > 0) and np.all(d.imag == 0) and np.array_equal(R, np.triu(R))
    if forward:
        Qo, Ro = O.qr_compact(A)
        assert np.linalg.norm(Q - Qo) <= 1e-12 * np.linalg.norm(Qo), A.shape
        assert np.linalg.norm(R - Ro) <= 1e-12 * np.linalg.norm(Ro), A.shape


@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
def test_whole_blocks_edges(dt, dev):
    """Packed and padded columns (odd leading dimensions) give the same
    factors; A is not written; nothing outside Q and R is written."""
    rng = np.random.default_rng(5)
    host = [conditioned(m, n, dt, 10.0 ** rng.uniform(0, 3), 50 + i) for i, (m, n) in enumerate(EDGE)]
    outs = []
    for pad in (0, 3):
        def view(m, n, fill):
            return torch.full((n, m + pad), fill, dtype=torch.float64 if dt == np.float64 else torch.complex128,
                              device=dev).t()
        bufs = [(view(m, n, 7.0), view(m, n, 7.0), view(n, n, 7.0)) for m, n in EDGE]
        for (a, _, _), h in zip(bufs, host):
            a[:h.shape[0]].copy_(torch.from_numpy(h).to(dev))
        views = [(a[:m], q[:m], r[:n]) for (a, q, r), (m, n) in zip(bufs, EDGE)]
        plan = mak.BatchedQRPlan([v[0] for v in views], [v[1] for v in views], [v[2] for v in views])
        plan.execute()
        torch.cuda.synchronize()
        outs.append([(q.cpu().numpy(), r.cpu().numpy()) for _, q, r in views])
        for (m, n), (a, q, r), h in zip(EDGE, bufs, host):
            if m >= 64:
                assert np.array_equal(a[:m].cpu().numpy(), h)
            for x, rows in ((q, m), (r, n)):
                assert (x[rows:] == 7.0).all()
        plan.close()
    for h, (q0, r0), (q1, r1) in zip(host, *outs):
        check(h, q0, r0, True)
        assert np.array_equal(q0, q1) and np.array_equal(r0, r1)


@pytest.mark.parametrize("with_r", [True, False])
@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
def test_whole_blocks_conditioning(dt, with_r, dev):
    """Condition numbers on both sides of the two bounds on ||Q1^H Q1 - I|| (one
    pass, two passes, left to the panels), a rank-deficient and a zero block,
    and values whose squares come near underflow; the graph replays with the same result
    after an execution on other values."""
    cases = [(150, 130, c) for c in (1e2, 1e4, 1e5, 3e5, 1e6, 1e8, 1e12)] + [(300, 70, 1e5), (90, 90, 1e5)]
    host = [conditioned(m, n, dt, c, 90 + i) for i, (m, n, c) in enumerate(cases)]
    host.append(conditioned(100, 80, dt, 1e2, 7) * 1e-150)
    D = conditioned(120, 90, dt, 1e2, 8)
    D[:, 70] = D[:, 3]
    special = [D, np.zeros((70, 66), dtype=dt)]
    As = [mak.colmajor(torch.from_numpy(np.asfortranarray(h)).to(dev)) for h in host + special]
    plan = mak.BatchedQRPlan(As) if with_r else mak.BatchedQRPlan(As, Rs=False)
    first = None
    for rep in range(3):
        for A, h in zip(As, host + special):
            A.copy_(torch.from_numpy(h if rep != 1 else conditioned(*h.shape, dt, 1e2, 3)).to(dev))
        Qs, Rs = plan.execute()
        torch.cuda.synchronize()
        if rep == 1:
            continue
        Qh = [q.cpu().numpy() for q in Qs]
        for h, q in zip(host, Qh):
            assert np.linalg.norm(q.conj().T @ q - np.eye(q.shape[1])) <= 1e-14 * np.sqrt(q.shape[1])
        if with_r:
            for h, q, r in zip(host, Qh, Rs):
                s = np.abs(h).max()  # powers of two apart, norms of squares near 1e-300 underflow
                check(h / s, q, r.cpu().numpy() / s, False)
        for q, h in zip(Qh[len(host):], special):
            assert np.linalg.norm(q.conj().T @ q - np.eye(q.shape[1])) <= 1e-14 * np.sqrt(q.shape[1])
        if first is None:
            first = Qh
        else:
            assert all(np.array_equal(a, b) for a, b in zip(first, Qh))
    plan.close()


@pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
def test_whole_blocks_rejected_in_the_middle_of_a_factor_step(dt, dev):
    """Blocks that lose positive definiteness at each of their diagonal tiles,
    while other tasks of the same block and other blocks are at work in the same
    launch: they come out as a QR of the block, and their neighbours as without
    them."""
    good = [O.gaussian(500, 450, dt, seed=60 + i) for i in range(4)]
    bad = []
    for t in range(1, 7):
        B = O.gaussian(460, 440, dt, seed=70 + t)
        B[:, 64 * t + 3] = B[:, 64 * t - 5]
        bad.append(B)
    outs = []
    for host in (good + 4 * bad, good):
        As = [mak.colmajor(torch.from_numpy(np.asfortranarray(h)).to(dev)) for h in host]
        plan = mak.BatchedQRPlan(As)
        Qs, Rs = plan.execute()
        torch.cuda.synchronize()
        outs.append([(q.cpu().numpy(), r.cpu().numpy()) for q, r in zip(Qs, Rs)])
        plan.close()
    for (q0, r0), (q1, r1), h in zip(outs[0], outs[1], good):
        assert np.array_equal(q0, q1) and np.array_equal(r0, r1)
        check(h, q0, r0, True)
    for h, (q, r) in zip(4 * bad, outs[0][4:]):
        assert np.linalg.norm(h - q @ r) <= 1e-14 * np.sqrt(h.shape[1]) * np.linalg.norm(h)
        assert np.linalg.norm(q.conj().T @ q - np.eye(q.shape[1])) <= 1e-14 * np.sqrt(q.shape[1])
