"""The default work shapes and the workgroup-per-item form of k_integrate: grids
of one bin, around the segment lengths and the groups of edges that a wavefront
loads ahead, a grid that lies inside the reach of the radii, one that the line
only touches at one end, redshifts, and batches on either side of the shapes'
bounds, against the oracle; and the same batch with a workgroup per item and
with persistent wavefronts.

Tolerances: 1e-8 (FP64) and 1e-4 (FP32) against the oracle, the bars of the
parity tests; two shapes of one batch add the same values in another order,
1e-12."""
import numpy as np
import pytest

import oracle
import relxill_amd as rx
from tests.helpers import RELLINE_CFG0, draw_relconv_params, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tabs():
    _, _, T = tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    return T


@pytest.mark.parametrize("band", [(0.1, 10.0), (5.0, 7.0), (6.0, 40.0), (0.05, 0.9)])
@pytest.mark.parametrize("n_bins", [1, 3, 4, 5, 7, 9, 31, 33, 65, 700, 2000, 9000])
def test_single_calls(tabs, n_bins, band):
    e = log_grid(n_bins, *band)
    for z in (0.0, 0.4):
        p = list(RELLINE_CFG0)
        p[8] = z
        ref, st = oracle.eval_model(oracle.MOD_RELLINE, tabs, p, e)
        for prec, tol in ((rx.FP64, 1e-8), (rx.FP32, 1e-4)):
            y, st_g = rx.eval_model(rx.MODEL_RELLINE, p, e, precision=prec)
            assert st == 0 and st_g == 0
            ok = np.isfinite(ref)
            np.testing.assert_array_equal(np.isfinite(y), ok)
            assert not ok.any() or rel_err(y[ok], ref[ok]) < tol


@pytest.mark.parametrize("n_req", [4, 5, 32, 33, 128, 129, 512, 513])
@pytest.mark.parametrize("prec", [0, 1])
def test_shapes_agree(tabs, n_req, prec):
    e = log_grid(150, 0.3, 9.0)
    reqs = []
    for q in draw_relconv_params(n_req, seed=n_req):
        reqs.append(dict(model=rx.MODEL_RELLINE, energy=e, params=[6.4, 3.0, 3.0, 15.0] + q[3:7] + [0.0, 0.0]))
    b = rx.Batch(reqs)
    outs = []
    for shape in ((0, 0), (150, 1), (1, 16), (64, 12)):
        b.set_shape(*shape)
        b.run(prec)
        b.sync()
        outs.append(np.array([b.output(i)[0] for i in range(n_req)]))
    b.close()
    for i in (0, n_req - 1):
        ref, st = oracle.eval_model(oracle.MOD_RELLINE, tabs, reqs[i]["params"], e)
        assert st == 0 and rel_err(outs[0][i], ref) < (1e-8 if prec == 0 else 1e-4)
    for o in outs[1:]:
        assert max(rel_err(o[i], outs[0][i]) for i in range(n_req)) < 1e-12
