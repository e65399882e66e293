"""The rotation as level-0 runs it (rot_quad: with and without mixed signs, and
the product of the norms that comes with it), bit for bit against the oracle at
the edges of its branches."""
import numpy as np
import pytest

import gpujachx_amd as g
import oracle as o

pytestmark = pytest.mark.gpu


def inputs():
    rng = np.random.default_rng(5)
    # zeta = z exactly: sqrt(eps/2), 1 and sqrt(2/eps) with their neighbours, zero,
    # subnormal, huge, infinite and NaN
    z = []
    for e in (float.fromhex("0x1.6a09e667f3bcdp-27"), 1.0, 2.0 ** 27):
        z += [e, np.nextafter(e, 0.0), np.nextafter(e, np.inf), e * (1.0 - 2.0 ** -30), e * (1.0 + 2.0 ** -30)]
    z += [0.0, 5e-324, 2.0 ** -1022, 1e-300, 0.5, 2.0, 1e300, np.finfo(float).max, np.inf, np.nan]
    z = np.array(z)
    cases = [(s * 0.5, dp, dq) for x in z for s in (1.0, -1.0) for dp, dq in ((0.0, x), (x, 0.0))]
    # nothing to rotate, equal columns, the ends of the range
    cases += [(0.0, 1.0, 1.0), (0.0, 1.0, 2.0), (-0.0, 2.0, 1.0), (0.0, 0.0, 0.0), (1e-320, 1.0, 1.0),
              (1e308, 1e308, 1e308), (np.inf, 1.0, 2.0), (np.nan, 1.0, 2.0), (1.0, 5e-324, 5e-324)]
    apq = rng.standard_normal(20000) * 10.0 ** rng.uniform(-18, 2, 20000)
    dp = 10.0 ** rng.uniform(-6, 6, 20000)
    dq = dp * (1.0 + 10.0 ** rng.uniform(-16, 3, 20000))
    dq[::2] = dp[::2] * (1.0 - 10.0 ** rng.uniform(-16, 0, 10000))
    a = np.array(cases)
    return np.r_[a[:, 0], apq], np.r_[a[:, 1], dp], np.r_[a[:, 2], dq]


@pytest.mark.parametrize("kind,fn", [(1, "rot_t"), (2, "rot_h"), (3, "rot_t")])
def test_rotation_of_level0(kind, fn):
    g.configureGPU(0)
    apq, dp, dq = inputs()
    c, t, big = g.dbg_scalar(kind, apq, dp, dq)
    ro = [getattr(o, fn)(*x) for x in zip(apq, dp, dq)]
    np.testing.assert_array_equal(c, [r[0] for r in ro])
    np.testing.assert_array_equal(t, [r[1] for r in ro])
    np.testing.assert_array_equal(big, [r[2] for r in ro])
    with np.errstate(all="ignore"):
        norms = np.sqrt(dp) * np.sqrt(dq)
    d, t2, big2 = g.dbg_scalar(kind + 3, apq, dp, dq)
    np.testing.assert_array_equal(d, norms)
    np.testing.assert_array_equal(t2, t)
    np.testing.assert_array_equal(big2, big)
