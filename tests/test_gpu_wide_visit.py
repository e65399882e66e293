"""The 64-column visit at the edges of its fast paths, bit for bit against the
oracle: pivots outside the range the short reciprocal square root takes, in the
first 32 columns of a pair (the general panel runs), in the last 32 (the general
32x32 Cholesky) or in both; signs that change anywhere in a pair; inner sweeps
to convergence; one and several row chunks."""
import numpy as np
import pytest

import gpujachx_amd as g
from test_gpu_wide import _both, assert_same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    g.configureGPU(0)
    old = g.lib().hj_set_block_width(32)
    yield
    g.lib().hj_set_block_width(old)


@pytest.mark.parametrize("scale", [-142.0, 142.0, -139.6, 139.8])
@pytest.mark.parametrize("cols", [slice(0, 32), slice(32, 64), slice(0, 64), slice(7, 40)])
@pytest.mark.parametrize("alg,nplus", [(11, 64), (8, 20)])
def test_pivots_beyond_the_short_root(scale, cols, alg, nplus):
    rng = np.random.default_rng(int(scale * 10) % 991)
    G = rng.standard_normal((128, 64))
    G[:, cols] *= 10.0 ** (scale + rng.uniform(-0.5, 0.5, 64)[cols])
    rg, ro = _both(alg, G, nplus)
    assert_same(rg, ro)


@pytest.mark.parametrize("nplus", [1, 31, 32, 33, 63])
@pytest.mark.parametrize("alg,m,n", [(3, 64, 64), (11, 192, 64), (9, 1088, 128), (10, 4096, 64)])
def test_signs_and_row_counts(nplus, alg, m, n):
    rng = np.random.default_rng(m + nplus)
    rg, ro = _both(alg, rng.standard_normal((m, n)) * 10.0 ** rng.uniform(-3, 3, n), nplus)
    assert_same(rg, ro)


# the Gram's tiles on waves of their own (1, 2 and 4 sub-chunks a chunk), one
# wave a sub-chunk beyond 1024 of them, updates of 64 .. 512 rows a workgroup, V
# beside the next visits over an odd number of steps
@pytest.mark.parametrize("m,n,fam", [(576, 192, "mmstep"), (2048, 128, "cycwor"), (4096, 128, "rowcyc"),
                                     (1024, 960, "mmstep"), (8192, 64, "cycwor"), (4096, 1024, "cycwor")])
def test_launches_of_a_step(m, n, fam):
    rng = np.random.default_rng(n)
    G = rng.standard_normal((m, n)) * 10.0 ** rng.uniform(-1, 1, n)
    rg, ro = _both(11, G, n // 3, fam=fam)
    assert_same(rg, ro)
