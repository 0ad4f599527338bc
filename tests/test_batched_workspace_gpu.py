"""The workspace of a batched plan: without the gauge it holds no whole blocks'
scratch, and a plan with the gauge that is given only that much runs on panels."""
import ctypes as C

import numpy as np
import pytest
import torch

import mak_mi355x as mak
from mak_mi355x import _lib
from oracle import mak_oracle as O

DTYPES = pytest.mark.parametrize("dt", [np.float64, np.complex128], ids=["f64", "c64"])
SHAPES = [(70, 64), (300, 200), (130, 130), (40, 20), (64, 1), (200, 300)] + [(256, 256)] * 20


def size(dt, positive, tune):
    lib = _lib.load()
    ms, ns = ((C.c_int * len(SHAPES))(*v) for v in zip(*SHAPES))
    b = C.c_size_t(0)
    assert lib.mak_qr_batched_plan_workspace_size(int(dt == np.complex128), len(SHAPES), ms, ns, positive, tune,
                                                  C.byref(b)) == 0
    return b.value


@DTYPES
def test_sizes(dt):
    lib = _lib.load()
    ms, ns = ((C.c_int * len(SHAPES))(*v) for v in zip(*SHAPES))
    b = C.c_size_t(0)
    for tune in (0, 1):
        assert lib.mak_qr_batched_workspace_size(int(dt == np.complex128), len(SHAPES), ms, ns, tune, C.byref(b)) == 0
        assert b.value == size(dt, 1, tune) >= size(dt, 0, tune)
    # W and U of the whole blocks alone are 2 n^2 elements each
    es = 8 if dt == np.float64 else 16
    assert size(dt, 1, 0) - size(dt, 0, 0) >= 20 * 2 * 256 * 256 * es


@pytest.mark.gpu
@DTYPES
@pytest.mark.parametrize("positive,given,whole,tune",
                         [(1, 1, 1, 0), (1, 0, 0, 0), (0, 0, 0, 0), (1, 1, 1, 1), (0, 0, 0, 1)])
def test_plan_at_its_limit(positive, given, whole, tune, dt, dev):
    """`given`: the size of which plan is given; a byte less is refused where no
    smaller layout is left.  Nothing after the workspace is written."""
    lib = _lib.load()
    host = [O.gaussian(m, n, dt, seed=i) for i, (m, n) in enumerate(SHAPES)]
    As = [mak.colmajor(torch.from_numpy(np.asfortranarray(h)).to(dev)) for h in host]
    Q, R = zip(*(mak.initialize_output_qr(A, False) for A in As))

    def arr(vals, t):
        return (t * len(As))(*vals)

    nb = size(dt, given, tune)
    ws = torch.full((nb + 4096,), 0x55, dtype=torch.uint8, device=dev)

    def create(nbytes):
        h = C.c_void_p(None)
        st = lib.mak_qr_batched_plan_create(
            C.byref(h), int(dt == np.complex128), len(As), arr([A.shape[0] for A in As], C.c_int),
            arr([A.shape[1] for A in As], C.c_int), arr([A.data_ptr() for A in As], C.c_void_p),
            arr([mak.api._ld(A) for A in As], C.c_int), arr([q.data_ptr() for q in Q], C.c_void_p),
            arr([mak.api._ld(q) for q in Q], C.c_int), arr([r.data_ptr() for r in R], C.c_void_p),
            arr([mak.api._ld(r) for r in R], C.c_int), positive, tune, ws.data_ptr(), nbytes)
        return st, h

    if not given:
        assert create(nb - 1)[0] == -14
    st, h = create(nb)
    assert st == 0
    assert lib.mak_qr_batched_execute(h, mak.api._stream(dev)) == 0
    torch.cuda.synchronize()
    lib.maktest_batched_routes.restype = C.c_int
    lib.maktest_batched_routes.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p]
    panels, blocks = (C.c_int * 3)(), (C.c_int * 3)()
    assert lib.maktest_batched_routes(h, panels, blocks) == 0
    assert (sum(blocks) > 0) == bool(whole)
    lib.mak_qr_batched_plan_destroy(h)
    assert torch.all(ws[nb:] == 0x55)
    for a, q, r in zip(host, Q, R):
        q, r = q.cpu().numpy(), r.cpu().numpy()
        # Householder QR's backward error and loss of orthogonality: a few sqrt(n) u
        assert np.linalg.norm(a - q @ r) <= 1e-14 * np.linalg.norm(a) * np.sqrt(a.shape[1])
        assert np.linalg.norm(q.conj().T @ q - np.eye(q.shape[1])) <= 1e-14 * q.shape[1]
