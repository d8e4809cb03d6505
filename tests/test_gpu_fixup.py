"""k_fixup: every queued re-check is done once, whatever the length of the queue:
one request by itself (few entries, idle lane groups) and 20 times in a batch
(several rounds over the workgroups), with and without emission-angle rows, on
narrow bins and on a convolution's wide ones.

The same values are added in another order: at most 16 chunks and as many
re-checks a bin, FP64: 1e-12 with margin."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import conv_err, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limb", [0, 1])
@pytest.mark.parametrize("model,n_bins,guard", [(rx.MODEL_RELLINE, 301, 5e-4), (rx.MODEL_RELLINE, 301, 0.95),
                                                (rx.MODEL_RELCONV, 500, 0.5)])
def test_queue_lengths(model, n_bins, guard, limb):
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    e = log_grid(n_bins, 0.5, 9.0)
    p = list(rx.DEFAULTS[model])
    line = model == rx.MODEL_RELLINE
    p[-1] = float(limb)
    req = dict(model=model, energy=e, params=p)
    if not line:
        req["flux_in"] = np.diff(e) / (0.5 * (e[1:] + e[:-1]))
    assert rx.lib.rx_set_fp32_guard(guard) == 0
    try:
        one, many = rx.Batch([req]), rx.Batch([req] * 20)
        for b in (one, many):
            b.run(rx.FP32)
            b.sync()
        n1, n2 = one.counters()["fp64_rechecks"], many.counters()["fp64_rechecks"]
        print(f"re-checks {n1} and {n2}", flush=True)
        assert n2 == 20 * n1 and (n1 > 0 or guard < 0.1) and many.counters()["recheck_overflow"] == 0
        ref = one.output(0)[0]
        for i in (0, 1, 10, 19):
            y, st = many.output(i)
            assert st == 0 and (rel_err(y, ref) if line else conv_err(y, ref)) < 1e-12
        one.close()
        many.close()
    finally:
        assert rx.lib.rx_set_fp32_guard(5e-4) == 0
