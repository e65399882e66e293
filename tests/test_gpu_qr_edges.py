"""The QR path of a visit at its edges, bit for bit against the oracle: the
fewest panels, a full set in LDS and one and many panels beyond it; entries
outside the range of plain sums of squares, in some columns or in all, cosines
formed from products out of range; zero columns and signs inside a block."""
import numpy as np
import pytest

import gpujachx_amd as g
import oracle as o
from test_gpu_qr import assert_same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    g.configureGPU(0)
    g.set_max_sweeps(4)
    o.set_max_sweeps(4)
    yield
    g.set_max_sweeps(30)
    o.set_max_sweeps(30)
    g.set_factorization(g.FACT_CHOLESKY)
    o.set_factorization(o.FACT_CHOLESKY)


def both(fact, alg, G, nplus):
    n = G.shape[1]
    g.init_strats_builtin("cycwor", 32, "mmstep", n // 16)
    s0, s1 = g.current_strats()
    g.set_factorization(fact)
    o.set_factorization(fact)
    try:
        rg = g.hypJacL2(alg, G, nplus)
        ro = o.hypJacL2(alg, G, nplus, s0, s1)
    finally:
        g.set_factorization(g.FACT_CHOLESKY)
        o.set_factorization(o.FACT_CHOLESKY)
    assert_same(rg, ro)


@pytest.mark.parametrize("fact", [g.FACT_QR, g.FACT_QR_DRMAC])
@pytest.mark.parametrize("m,n", [(64, 32), (64, 64), (128, 96), (448, 32), (512, 64), (576, 64), (960, 32), (1024, 64), (1536, 32)])
def test_panel_counts(fact, m, n):
    rng = np.random.default_rng(m + n)
    G = rng.standard_normal((m, n)) * 10.0 ** rng.uniform(-8, 8, n)
    both(fact, 11, G, n)
    both(fact, 8, G, n // 3)


@pytest.mark.parametrize("alg,nplus", [(11, 64), (11, 0), (1, 64), (9, 21)])
@pytest.mark.parametrize("lo,hi", [(-175, -150), (-158, -150), (150, 155), (-160, 150), (-170, 10)])
def test_magnitudes_beyond_plain_sums(lo, hi, alg, nplus):
    rng = np.random.default_rng(hi - lo)
    G = rng.standard_normal((128, 64)) * 10.0 ** rng.uniform(lo, hi, 64)
    G[:, ::7] *= 10.0 ** rng.uniform(-6, 0, (128, 10))
    both(g.FACT_QR_DRMAC, alg, G, nplus)
    both(g.FACT_QR, alg, G, nplus)


@pytest.mark.parametrize("alg", [11, 8])
def test_dependent_and_sparse_columns(alg):
    rng = np.random.default_rng(4)
    G = rng.standard_normal((192, 64))
    G[:, 5] = 0.0
    G[:, 40] = G[:, 39]          # a cosine of one: the cotangent overflows
    G[32:, 17] = 0.0             # panels with a zero column
    G[:160, 20] = 0.0
    both(g.FACT_QR_DRMAC, alg, G, 64)
