"""mak_qr_compact_noalloc_d one call after the other on two streams: the calls
share one static scratch array, and each is over when it returns, on every path
(positive = False and matrices under 64 rows enqueue work without a read at their
end).  The results are the workspace entry point's, bit for bit."""
import ctypes as C

import numpy as np
import pytest
import torch

import mak_mi355x as mak
from mak_mi355x import _lib
from oracle import mak_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,positive", [(60, 40, 1), (1000, 300, 0), (900, 40, 0), (600, 200, 1)])
def test_calls_in_turn_on_two_streams(m, n, positive, dev):
    lib = _lib.load()
    As = [mak.colmajor(torch.from_numpy(np.asfortranarray(O.gaussian(m, n, np.float64, seed=i))).to(dev))
          for i in range(8)]
    refs = [mak.qr_compact(A, mak.MI355XHouseholder(positive=bool(positive))) for A in As]
    outs = [mak.initialize_output_qr(A, False) for A in As]
    copies = [A.clone() for A in As]
    streams = [torch.cuda.Stream(dev) for _ in range(2)]
    torch.cuda.synchronize()
    for i, (A, (Q, R)) in enumerate(zip(copies, outs)):
        s = streams[i % 2]
        assert lib.mak_qr_compact_noalloc_d(C.c_void_p(s.cuda_stream), m, n, C.c_void_p(A.data_ptr()), m,
                                            C.c_void_p(Q.data_ptr()), m, C.c_void_p(R.data_ptr()), n, positive) == 0
        assert s.query()
    torch.cuda.synchronize()
    for (Q, R), (Qr, Rr) in zip(outs, refs):
        assert torch.equal(Q, Qr) and torch.equal(R, Rr)
