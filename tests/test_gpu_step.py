"""The launches of a small step, bit for bit against the oracle, at the sizes
where the choice between them changes: the whole step in one launch (up to 512
rows of G and V together), the Gram's tiles on waves of their own (few
sub-chunks of 1, 2 or 4 waves a chunk), V updated beside the next step's visits,
and transitions that are closed but not fused."""
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
    g.set_max_sweeps(30)


def both(alg, m, n, nplus, fam, limit=0, seed=3):
    rng = np.random.default_rng(seed)
    G = rng.standard_normal((m, n)) * 10.0 ** rng.uniform(-3, 3, n)
    g.init_strats_builtin("cycwor", 32, fam, n // 16)
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


# one launch a step: 1 (all odd multiples of 64), 2, 4 and 8 sub-chunks; the
# last rows of its range and the first beyond it, with and without V
@pytest.mark.parametrize("alg,m,n", [(11, 64, 32), (9, 64, 64), (11, 128, 64), (10, 192, 96), (11, 256, 256),
                                     (3, 320, 64), (11, 384, 128), (8, 448, 64), (9, 512, 128), (11, 512, 32),
                                     (11, 320, 192), (11, 320, 224)])
def test_whole_step(alg, m, n):
    both(alg, m, n, n // 3, "mmstep")


# Gram tiles: one wave a chunk over 9 .. 21 panels, two and four waves; the
# first of the plain kernel's range (512 sub-chunks and more)
@pytest.mark.parametrize("m,n,limit", [(576, 64, 0), (1088, 64, 0), (1344, 96, 0), (2048, 32, 0), (4096, 64, 0),
                                       (6144, 64, 3), (2048, 512, 2), (2048, 544, 2)])
def test_gram_tiles(m, n, limit):
    both(9, m, n, n, "mmstep", limit)


# V beside the next visits: a run ended inside a sweep, at its end, and over
# several sweeps; fused and unfused transitions
@pytest.mark.parametrize("m,n,fam,limit", [(1024, 256, "cycwor", 1), (1024, 256, "cycwor", 2),
                                           (1024, 256, "cycwor", 17), (1024, 256, "rowcyc", 0),
                                           (2048, 1024, "cycwor", 3), (4096, 1024, "cycwor", 4),
                                           (640, 480, "BrentL", 31)])
def test_v_rides_with_the_next_visits(m, n, fam, limit):
    both(11, m, n, n // 2, fam, limit)


# sweeps queued one ahead (one launch a step), or not (three): ended by the cap
# or by convergence, at every parity, twice in a row
@pytest.mark.parametrize("cap", [1, 2, 3, 4, 30])
@pytest.mark.parametrize("alg,m,n", [(11, 64, 32), (9, 128, 64), (2, 256, 96), (11, 1024, 96), (9, 2048, 224)])
def test_sweeps_queued_ahead(cap, alg, m, n):
    rng = np.random.default_rng(cap)
    G = rng.standard_normal((m, n))
    g.init_strats_builtin("cycwor", 32, "mmstep", n // 16)
    s0, s1 = g.current_strats()
    g.set_max_sweeps(cap)
    o.set_max_sweeps(cap)
    try:
        ro = o.hypJacL2(alg, G, n, s0, s1)
        for _ in range(2):
            rg = g.hypJacL2(alg, G, n)
            assert (rg.sweeps, rg.rot_s, rg.rot_b) == (ro["sweeps"], ro["rot_s"], ro["rot_b"])
            np.testing.assert_array_equal(rg.D, ro["D"])
            np.testing.assert_array_equal(rg.G, ro["G"])
    finally:
        g.set_max_sweeps(30)
        o.set_max_sweeps(30)


# the same without allocation (the scratch array is used again)
@pytest.mark.parametrize("cap", [1, 2, 3, 30])
@pytest.mark.parametrize("m,n", [(64, 32), (576, 64), (2048, 128)])
def test_noalloc_sweep_caps(cap, m, n):
    import ctypes
    import torch
    rng = np.random.default_rng(cap)
    G = np.asfortranarray(rng.standard_normal((m, n)))
    g.init_strats_builtin("cycwor", 32, "mmstep", n // 16)
    s0, s1 = g.current_strats()
    g.set_max_sweeps(cap)
    o.set_max_sweeps(cap)
    try:
        ro = o.hypJacL2(11, G, n, s0, s1)
        for _ in range(2):
            dG = torch.from_numpy(G.T.copy()).cuda()
            dV, dD = torch.zeros(n, n, dtype=torch.float64, device="cuda"), torch.zeros(n, dtype=torch.float64, device="cuda")
            sw, gs, gb = ctypes.c_uint(0), ctypes.c_ulonglong(0), ctypes.c_ulonglong(0)
            rc = g.lib().hypJacL2_dev_noalloc(11, m, n, n, dG.data_ptr(), m, dV.data_ptr(), n, dD.data_ptr(),
                                              ctypes.byref(sw), ctypes.byref(gs), ctypes.byref(gb), None,
                                              torch.cuda.current_stream().cuda_stream)
            assert rc == 0 and (sw.value, gs.value, gb.value) == (ro["sweeps"], ro["rot_s"], ro["rot_b"])
            np.testing.assert_array_equal(dD.cpu().numpy(), ro["D"])
            np.testing.assert_array_equal(dG.cpu().numpy().T, ro["G"])
            np.testing.assert_array_equal(dV.cpu().numpy().T, ro["V"])
    finally:
        g.set_max_sweeps(30)
        o.set_max_sweeps(30)
