"""One step of the thin level-1 layer with more pairs than the chip has CUs: 512
rows of more than 256 pairs are Gram chunks of 128 rows, two waves each, which
the one-launch step does not form.  Every pair bit for bit against the oracle."""
import ctypes

import numpy as np
import pytest
import torch

import gpujachx_amd as g
import oracle as o
from test_gpu_thin import _bind

pytestmark = pytest.mark.gpu


# the last order with chunks of one wave (256 pairs) and the next of the table
@pytest.mark.parametrize("m,n", [(512, 8192), (512, 8224), (448, 8224)])
def test_one_step(m, n):
    g.configureGPU(0)
    L, lo = _bind(), o.lib()
    rng = np.random.default_rng(n)
    Gt = rng.standard_normal((n, m)) * 10.0 ** rng.uniform(-3, 3, (n, 1))
    g.init_strats_builtin("cycwor", 32, "mmstep", n // 16)
    s0, s1 = g.current_strats()
    s0 = np.ascontiguousarray(s0, dtype=np.uint8)
    Gd = torch.from_numpy(Gt.copy()).cuda()
    cvg = torch.zeros(1, dtype=torch.int64, device="cuda")
    L.initSymbols(Gd.data_ptr(), None, cvg.data_ptr(), m, n, m, 0, 1)
    L.defJacL1s(0, 1)
    torch.cuda.synchronize()
    got = Gd.cpu().numpy()
    pd = ctypes.POINTER(ctypes.c_double)

    def at(a, i=0):
        return ctypes.cast(a.ctypes.data + 8 * i, pd)
    nc = o.gram_nchunk(m, n // 32)
    ch = m // nc
    for i, j in s1[0].astype(int):
        cols = np.r_[16 * i:16 * i + 16, 16 * j:16 * j + 16]
        P = np.ascontiguousarray(Gt[cols])
        part = np.zeros((nc, 768))
        for c in range(nc):
            lo.hjo_gram_partial(at(P), at(P, 16 * m), m, c * ch, ch, at(part, 768 * c))
        W, _, _, _, upd = o.pair(part, 1, 0, 1, 0, s0)
        if upd:
            Wc = np.ascontiguousarray(W.T)
            lo.hjo_update(at(P), at(P, 16 * m), m, m, at(Wc))
        np.testing.assert_array_equal(got[cols], P, err_msg="blocks %d, %d" % (i, j))
