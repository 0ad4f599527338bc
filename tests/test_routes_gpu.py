"""Which path a factorisation took: the CholeskyQR2 forms for inputs far inside
what they accept, the Householder forms for inputs far outside it, and the
panels that run under each.  The other tests check results, which every path
meets; these fail when a path is not taken."""
import ctypes as C

import numpy as np
import pytest
import torch

import mak_mi355x as mak
from mak_mi355x import _lib
from oracle import mak_oracle as O

pytestmark = pytest.mark.gpu
DTYPES = pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])


def conditioned(m, n, dt, cond, seed):
    """m x n with singular values log-spaced from 1 to 1 / cond."""
    rng = np.random.default_rng(seed)

    def ortho(r, c):
        x = rng.standard_normal((r, c))
        if dt == np.complex128:
            x = x + 1j * rng.standard_normal((r, c))
        return np.linalg.qr(x)[0]

    return (ortho(m, n) * np.logspace(0, -np.log10(cond), n)) @ ortho(n, n).conj().T


def to_dev(A, dev):
    return mak.colmajor(torch.from_numpy(np.asfortranarray(A)).to(dev))


def run_record(A, dev, full=False, positive=True, words=False):
    """Q, R and whether the whole matrix's CholeskyQR2 was accepted (words: the
    whole record)."""
    At = to_dev(A, dev)
    m, n = At.shape
    Q, R = mak.initialize_output_qr(At, full)
    lib = _lib.load()
    dt = 1 if At.is_complex() else 0
    nb = C.c_size_t(0)
    assert lib.mak_qr_workspace_size(dt, int(full), m, n, C.byref(nb)) == 0
    ws = torch.full((nb.value,), 0x55, dtype=torch.uint8, device=dev)
    f = getattr(lib, f"mak_qr_{'full' if full else 'compact'}_{'z' if dt else 'd'}")
    assert f(mak.api._stream(dev), m, n, mak.api._ptr(At), mak.api._ld(At), mak.api._ptr(Q), mak.api._ld(Q),
             mak.api._ptr(R), mak.api._ld(R), int(positive), mak.api._ptr(ws), nb.value) == 0
    torch.cuda.synchronize()
    lib.maktest_qr_record.restype = C.c_int
    lib.maktest_qr_record.argtypes = [C.c_int, C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    rec = (C.c_int * 9)()
    assert lib.maktest_qr_record(dt, int(full), m, n, C.c_void_p(ws.data_ptr()), rec) == 0
    return Q.cpu().numpy(), R.cpu().numpy(), list(rec) if words else rec[0]


def routes(plan):
    """Panels (accepted, rejected, not run) and whole blocks (one pass, two
    passes, rejected) of the plan's last execution."""
    lib = _lib.load()
    lib.maktest_batched_routes.restype = C.c_int
    lib.maktest_batched_routes.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p]
    panels, whole = (C.c_int * 3)(), (C.c_int * 3)()
    assert lib.maktest_batched_routes(plan._h, panels, whole) == 0
    return tuple(panels), tuple(whole)


def sound(A, Q, R):
    assert np.linalg.norm(A - Q @ R) <= 1e-14 * np.sqrt(A.shape[1]) * np.linalg.norm(A)
    assert np.linalg.norm(Q.conj().T @ Q - np.eye(Q.shape[1])) <= 1e-14 * Q.shape[1]


@DTYPES
@pytest.mark.parametrize("m,n", [(20, 7), (57, 33), (63, 63), (64, 1), (70, 63), (700, 40), (16384, 33), (300, 64)])
def test_compact_routes(m, n, dt, dev):
    for cond, taken in ((1.0, 1), (1e2, 1), (1e12, 0)):
        if n == 1 and cond > 1:
            continue
        A = conditioned(m, n, dt, cond, m + n)
        Q, R, got = run_record(A, dev)
        assert got == taken, cond
        sound(A, Q, R)


@DTYPES
@pytest.mark.parametrize("full,positive", [(True, True), (True, False), (False, False)])
@pytest.mark.parametrize("m,n", [(200, 64), (400, 150)])
def test_signed_and_full_routes(m, n, full, positive, dt, dev):
    for cond, taken in ((1e2, 1), (1e12, 0)):
        A = conditioned(m, n, dt, cond, m + n)
        Q, R, got = run_record(A, dev, full, positive)
        assert got == taken, cond
        sound(A, Q, R)


@DTYPES
@pytest.mark.parametrize("m,n", [(4000, 200), (3000, 290)])
def test_paired_block_reflectors_of_a_rejected_input(m, n, dt, dev):
    """qr_full! whose Q is formed by 256-column block reflectors: a full group
    of 128 columns paired with one of 72, and a third group left unpaired."""
    A = conditioned(m, n, dt, 1e12, m)
    Q, R, got = run_record(A, dev, full=True)
    assert got == 0
    Qt, At = torch.from_numpy(Q).to(dev), torch.from_numpy(A).to(dev)
    eye = torch.eye(m, dtype=Qt.dtype, device=dev)
    assert (torch.linalg.norm(Qt.mH @ Qt - eye) / np.sqrt(m)).item() < 1e-13
    assert (torch.linalg.norm(At - Qt @ torch.from_numpy(R).to(dev)) / torch.linalg.norm(At)).item() < 1e-13
    assert np.all(np.tril(R, -1) == 0)


@DTYPES
def test_whole_block_routes(dt, dev):
    """One pass for condition 1e2, two for 1e6, the panels for 1e12; the panels
    of blocks that were factored whole do not run."""
    for cond, want in ((1e2, (3, 0, 0)), (1e6, (0, 3, 0)), (1e12, (0, 0, 3))):
        host = [conditioned(m, n, dt, cond, m) for m, n in ((150, 130), (400, 64), (90, 90))]
        plan = mak.BatchedQRPlan([to_dev(h, dev) for h in host])
        Qs, Rs = plan.execute()
        torch.cuda.synchronize()
        panels, whole = routes(plan)
        assert whole == want, cond
        count = sum(1 for h in host for j in range(0, h.shape[1], 32) if h.shape[0] - j >= 64)
        assert sum(panels) == count and panels[2] == (0 if want[2] else count)
        for h, q, r in zip(host, Qs, Rs):
            sound(h, q.cpu().numpy(), r.cpu().numpy())
        plan.close()


@DTYPES
def test_panels_of_a_plan_without_the_gauge(dt, dev):
    """positive = False keeps every block on panels: all of at least 64 rows are
    factored by their CholeskyQR2 task for Gaussian blocks."""
    shapes = mak.block_shapes(120, seed=9, mmax=1000)
    host = [O.gaussian(m, n, dt, seed=300 + i) for i, (m, n) in enumerate(shapes)]
    plan = mak.BatchedQRPlan([to_dev(h, dev) for h in host], alg=mak.MI355XHouseholder(positive=False))
    Qs, Rs = plan.execute()
    torch.cuda.synchronize()
    count = sum(1 for m, n in shapes for j in range(0, min(m, n), 32) if m - j >= 64)
    assert routes(plan) == ((count, 0, 0), (0, 0, 0))
    for i in range(0, 120, 17):
        sound(host[i], Qs[i].cpu().numpy(), Rs[i].cpu().numpy())
    plan.close()


@DTYPES
@pytest.mark.parametrize("m,n", [(500, 100), (2100, 1024)])
@pytest.mark.parametrize("full,positive", [(True, True), (True, False), (False, False)])
def test_signed_and_full_run_on_fp64(m, n, full, positive, dt, dev):
    """Only qr_compact! with positive = True may form its final correction on BF16
    or FP32 MFMA (record: FP32, FP64, BF16 in words 6 to 8)."""
    A = O.gaussian(m, n, dt, seed=11)
    assert run_record(A, dev, full, positive, words=True)[2][6:9] == [0, 1, 0]


@DTYPES
def test_small_compact_is_the_full_factorisation(dt, dev):
    """Below the size where the low-precision correction is faster, qr_compact! and
    qr_full! run the same FP64 products: the same bits."""
    for m, n in ((100, 64), (900, 200)):
        A = to_dev(O.gaussian(m, n, dt, seed=12), dev)
        (Qc, Rc), (Qf, Rf) = mak.qr_compact(A), mak.qr_full(A)
        assert torch.equal(Qc, Qf[:, :n]) and torch.equal(Rc, Rf[:n])
