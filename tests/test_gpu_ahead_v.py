"""Sweeps queued one ahead (one launch a step) and V: the sweep queued after the
last one leaves it as it is, whether the cap or convergence ended the run, at
every parity and twice in a row."""
import numpy as np
import pytest

import gpujachx_amd as g
import oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [1, 2, 3, 30])
@pytest.mark.parametrize("alg,m,n,nplus", [(11, 64, 32, 32), (2, 192, 96, 96), (11, 256, 256, 100), (10, 320, 192, 0)])
def test_v_after_the_last_sweep(cap, alg, m, n, nplus):
    g.configureGPU(0)
    rng = np.random.default_rng(cap + n)
    # columns nearly in order and nearly orthogonal: convergence within the caps
    G = np.linalg.qr(rng.standard_normal((m, n)))[0] * np.arange(n, 0.0, -1.0) + 1e-6 * rng.standard_normal((m, n))
    g.init_strats_builtin("cycwor", 32, "mmstep", n // 16)
    s0, s1 = g.current_strats()
    g.set_max_sweeps(cap)
    o.set_max_sweeps(cap)
    try:
        ro = o.hypJacL2(alg, G, nplus, s0, s1)
        for _ in range(2):
            rg = g.hypJacL2(alg, G, nplus)
            assert (rg.sweeps, rg.rot_s, rg.rot_b) == (ro["sweeps"], ro["rot_s"], ro["rot_b"])
            np.testing.assert_array_equal(rg.V, ro["V"])
            np.testing.assert_array_equal(rg.G, ro["G"])
    finally:
        g.set_max_sweeps(30)
        o.set_max_sweeps(30)
