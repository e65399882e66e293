"""The thin level-1 layer at row counts that 32 divides and 64 does not, bit for
bit against the oracle on the matrix with zero rows below (they add nothing to
its one Gram chain over the rows, to a column norm or to any other row)."""
import numpy as np
import pytest
import torch

import gpujachx_amd as g
import oracle as o
from test_gpu_thin import _bind

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    g.configureGPU(0)
    yield
    o.set_single_wave_gram(False)
    o.set_factorization(0)
    g.set_factorization(g.FACT_CHOLESKY)


def one_sweep(m, n, alg, nplus, fact=0):
    L = _bind()
    rng = np.random.default_rng(m + n)
    G = rng.standard_normal((m, n)) * 10.0 ** rng.uniform(-3, 3, n)
    g.init_strats_builtin("cycwor", 32, "mmstep", n // 16)
    s0, s1 = g.current_strats()
    full = bool(alg & 2)
    Gd = torch.from_numpy(G.T.copy()).cuda()
    Vd = torch.zeros((n, n), dtype=torch.float64, device="cuda") if full else None
    Dd = torch.zeros(n, dtype=torch.float64, device="cuda")
    cvg = torch.zeros(1, dtype=torch.int64, device="cuda")
    g.set_factorization(fact)
    L.initSymbols(Gd.data_ptr(), Vd.data_ptr() if full else None, cvg.data_ptr(), m, n, m, n if full else 0, 1)
    if full:
        L.initV(Vd.data_ptr(), 0, n, n)
    fn = getattr(L, ("def" if nplus == n else "hyp") + "JacL1" + ("s" if alg & 1 else "") + ("v" if full else ""))
    for st in range(s1.shape[0]):
        fn(st, 1 if nplus == n else nplus)
    L.initD(Gd.data_ptr(), Dd.data_ptr(), 0, m, n, nplus, m)
    torch.cuda.synchronize()
    g.set_factorization(g.FACT_CHOLESKY)
    pad = np.zeros((m + 32, n))
    pad[:m] = G
    o.set_single_wave_gram(True)
    o.set_factorization(fact)
    try:
        ro = o.hypJacL2(alg, pad, nplus, s0, s1, max_steps=s1.shape[0])
    finally:
        o.set_single_wave_gram(False)
        o.set_factorization(0)
    assert ro["ret"] == 0 and not ro["G"][m:].any()
    np.testing.assert_array_equal(Gd.cpu().numpy().T, ro["G"][:m])
    np.testing.assert_array_equal(Dd.cpu().numpy(), ro["D"])
    if full:
        np.testing.assert_array_equal(Vd.cpu().numpy().T, ro["V"])
    c = int(cvg.cpu().numpy()[0])
    assert (c & 0xFFFFFFFF, c >> 32) == (ro["rot_s_trace"][0], ro["rot_b_trace"][0])


# one 32-row group and more, odd and even numbers of 64 rows before the last 32;
# around the whole step's 512 rows, with and without V
@pytest.mark.parametrize("m,n,alg", [(32, 32, 9), (32, 32, 11), (96, 64, 11), (160, 64, 9), (160, 96, 11), (224, 32, 8),
                                     (480, 32, 11), (480, 64, 9), (544, 64, 11), (1056, 96, 10)])
@pytest.mark.parametrize("hyp", [False, True])
def test_thin_rows(m, n, alg, hyp):
    one_sweep(m, n, alg, n // 3 if hyp else n)


@pytest.mark.parametrize("fact", [1, 2])
@pytest.mark.parametrize("m,n", [(32, 32), (96, 64), (544, 64)])
def test_thin_rows_qr(m, n, fact):
    one_sweep(m, n, 11, n, fact)
