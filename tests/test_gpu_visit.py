"""The pair visit at the edges of its fast paths, bit for bit against the
oracle: pivots outside the range the short reciprocal square root takes (the
general Cholesky runs), mixed with pivots inside it; zero columns; inner
sweeps to convergence; signs that change inside a block."""
import numpy as np
import pytest

import gpujachx_amd as g
import oracle as o

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    g.configureGPU(0)
    yield
    g.set_step_limit(0)


def both(alg, G, nplus, limit=0):
    n = G.shape[1]
    g.init_strats_builtin("cycwor", 32, "cycwor", n // 16)
    s0, s1 = g.current_strats()
    g.set_step_limit(limit)
    try:
        rg = g.hypJacL2(alg, G, nplus)
    finally:
        g.set_step_limit(0)
    ro = o.hypJacL2(alg, G, nplus, s0, s1, max_steps=limit)
    assert rg.ret == 0 and ro["ret"] == 0
    assert (rg.sweeps, rg.rot_s, rg.rot_b) == (ro["sweeps"], ro["rot_s"], ro["rot_b"])
    np.testing.assert_array_equal(rg.D, ro["D"])
    np.testing.assert_array_equal(rg.G, ro["G"])
    if ro["V"] is not None:
        np.testing.assert_array_equal(rg.V, ro["V"])


@pytest.mark.parametrize("lo,hi", [(-142.0, -142.0), (142.0, 142.0), (-145.0, 145.0), (-140.5, -138.5),
                                   (139.0, 140.5)])
@pytest.mark.parametrize("alg,nplus", [(11, 64), (9, 23), (2, 64)])
def test_column_scales_beyond_the_short_root(lo, hi, alg, nplus):
    rng = np.random.default_rng(int(lo * 10) % 997 + alg)
    G = rng.standard_normal((128, 64)) * 10.0 ** rng.uniform(lo, hi, 64)
    both(alg, G, nplus)


@pytest.mark.parametrize("alg", [11, 8])
@pytest.mark.parametrize("zeros", [[5], [0, 31], [16, 17, 40]])
def test_zero_columns_two_steps(alg, zeros):
    rng = np.random.default_rng(7)
    G = rng.standard_normal((128, 64))
    G[:, zeros] = 0.0
    both(alg, G, 64, limit=2)


@pytest.mark.parametrize("nplus", [1, 15, 17, 31, 33, 63])
@pytest.mark.parametrize("alg", [3, 11, 8])
def test_sign_change_inside_a_block(nplus, alg):
    rng = np.random.default_rng(nplus)
    both(alg, rng.standard_normal((192, 64)) * 10.0 ** rng.uniform(-3, 3, 64), nplus)
