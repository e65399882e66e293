"""The launch shape of a batch: a configuration's own, whatever it is, and the
plan's choice only without a configuration; every shape's results bit for bit
those of the oracle."""
import numpy as np
import pytest
import torch

import gpujachx_amd as g
import oracle as o
from test_gpu_batch import SHAPES, _oracle, _problems

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    g.configureGPU(0)
    yield
    o.set_single_wave_gram(False)


def _on_device(probs):
    keep, descs = [], []
    for G, nplus, alg in probs:
        m, n = G.shape
        Gd = torch.from_numpy(G.T.copy()).cuda()
        Dd = torch.zeros(n, dtype=torch.float64, device="cuda")
        Vd = torch.zeros((n, n), dtype=torch.float64, device="cuda") if alg & 2 else None
        keep.append((Gd, Vd, Dd))
        descs.append(g.BatchDesc(alg, m, n, nplus, m, n if Vd is not None else 0, Gd.data_ptr(),
                                 Vd.data_ptr() if Vd is not None else None, Dd.data_ptr()))
    return keep, descs


# None: the plan's choice.  For these twelve problems on 256 CUs the largest one
# (512 x 320, ten pairs a step) ends the run, and eight waves end it first.
@pytest.mark.parametrize("shape", [(4, 2), (8, 1), (2, 4), None])
def test_shape_that_runs(shape):
    probs = _problems(31, SHAPES)
    keep, descs = _on_device(probs)
    cfg = None
    if shape:
        cfg = g.default_batch_cfg()
        cfg.waves, cfg.wg_per_cu = shape
    b = g.Batch(descs, cfg)
    try:
        assert b.shape() == (shape or (8, 1))
        b.run()
        res = b.results()
    finally:
        b.close()
    for k, ((G, nplus, alg), (Gd, Vd, Dd)) in enumerate(zip(probs, keep)):
        n1 = G.shape[1] // 16
        ro = _oracle(G, nplus, alg, "BrentL" if n1 & (n1 - 1) else "cycwor", 30)
        ctx = "problem %d %s alg %d shape %s" % (k, G.shape, alg, shape)
        assert (res["sweeps"][k], res["rot_s"][k], res["rot_b"][k]) == (ro["sweeps"], ro["rot_s"], ro["rot_b"]), ctx
        np.testing.assert_array_equal(Gd.cpu().numpy().T, ro["G"], err_msg=ctx)
        np.testing.assert_array_equal(Dd.cpu().numpy(), ro["D"], err_msg=ctx)
        if Vd is not None:
            np.testing.assert_array_equal(Vd.cpu().numpy().T, ro["V"], err_msg=ctx)


# the default configuration is a shape like any other, and a tuned one runs as
# it was timed
def test_default_and_tuned_shapes_are_kept():
    _, descs = _on_device(_problems(32, SHAPES))
    for cfg in (g.default_batch_cfg(), g.batch_autotune(descs, sample=6)[0]):
        b = g.Batch(descs, cfg)
        try:
            assert b.shape() == (cfg.waves, cfg.wg_per_cu)
        finally:
            b.close()
    assert (g.default_batch_cfg().waves, g.default_batch_cfg().wg_per_cu) == (4, 2)
