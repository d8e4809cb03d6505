"""Default segments of batches of 5 to 128 requests, which follow the bins that
the requests' windows can reach: on either side of each length, against the
oracle and against segments of other lengths.

Tolerances: 1e-8 (FP64) and 1e-4 (FP32) against the oracle, the bars of the
parity tests; two shapes of one batch add the same values in another order,
1e-12."""
import numpy as np
import pytest

import oracle
import relxill_amd as rx
from tests.helpers import draw_relconv_params, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


# about 450 thousand, 1 million and 4 million reachable bins are the bounds
@pytest.mark.parametrize("n_req,n_bins", [(5, 7000), (5, 9000), (12, 7000), (12, 8500), (33, 10500), (47, 7500), (32, 16384), (32, 16385)])
@pytest.mark.parametrize("prec", [0, 1])
def test_segments(n_req, n_bins, prec):
    _, _, T = tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    e = log_grid(n_bins, 0.1, 10.0)
    reqs = [dict(model=rx.MODEL_RELLINE, energy=e, params=[6.4, 3.0, 3.0, 15.0] + q[3:7] + [0.0, 0.0])
            for q in draw_relconv_params(n_req, seed=n_bins)]
    b = rx.Batch(reqs)
    outs = []
    for shape in ((0, 0), (8, 0), (256, 0)):
        b.set_shape(*shape)
        b.run(prec)
        b.sync()
        outs.append([b.output(i)[0] for i in range(n_req)])
    b.close()
    ref, st = oracle.eval_model(oracle.MOD_RELLINE, T, reqs[-1]["params"], e)
    assert st == 0 and rel_err(outs[0][-1], ref) < (1e-8 if prec == 0 else 1e-4)
    for o in outs[1:]:
        assert max(rel_err(o[i], outs[0][i]) for i in range(n_req)) < 1e-12
