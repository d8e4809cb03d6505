"""Results delivered by a run's last kernel: outputs and statuses of single calls
against the output array of a batch, for every kind of last kernel (line models,
one-zone convolutions with and without a primary, several zones, the xillver
models), and statuses of batches of each kind with a failing request between
good ones.

Line models add radius chunks in any order, 16 FP64 terms: 1e-12 with margin;
convolved spectra in faint bins: the suite's 1e-8 (conv_err)."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import conv_err, log_grid, tables

pytestmark = pytest.mark.gpu

LINE, CONV = (rx.MODEL_RELLINE, rx.MODEL_RELLINELP), (rx.MODEL_RELCONV, rx.MODEL_RELCONVLP)
OTHER = (rx.MODEL_RELXILL, rx.MODEL_RELXILLLP, rx.MODEL_RELXILLLPCP, rx.MODEL_XILLVER)


@pytest.fixture(scope="module")
def small_tables():
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    rx.xilltable_synthetic(5, 4, 3, 4, 3, 10, 300)
    rx.xillcptable_synthetic(6, 4, 3, 4, 3, 10, 300)
    yield
    rx.xilltable_synthetic()
    rx.xillcptable_synthetic()


def request(model, e, bad=False):
    p = list(rx.DEFAULTS[model])
    if bad:  # the inner disk edge beyond the outer one
        p[{rx.MODEL_RELLINE: 6, rx.MODEL_RELCONV: 5, rx.MODEL_RELXILL: 5}[model]] = 900.0
    r = dict(model=model, energy=e, params=p)
    if model in CONV:
        r["flux_in"] = np.diff(e) / (0.5 * (e[1:] + e[:-1]))
    return r


@pytest.mark.parametrize("precision", [rx.FP64, rx.FP32])
@pytest.mark.parametrize("model", LINE + CONV + OTHER)
def test_call_and_batch(small_tables, model, precision):
    e = log_grid(701, 0.2, 50.0)
    r = request(model, e)
    b = rx.Batch([r])
    b.run(precision)
    b.sync()
    ref, st = b.output(0)
    b.close()
    y, st1 = rx.eval_model(model, r["params"], e, r.get("flux_in"), precision=precision)
    assert st == 0 and st1 == 0 and np.any(ref > 0)
    if model in LINE:
        np.testing.assert_allclose(y, ref, rtol=1e-12, atol=1e-14 * ref.max())
    else:
        assert conv_err(y, ref) < 1e-8


@pytest.mark.parametrize("model", [rx.MODEL_RELLINE, rx.MODEL_RELCONV, rx.MODEL_RELXILL])
def test_statuses(small_tables, model):
    e = log_grid(300, 0.2, 50.0)
    reqs = [request(model, e, bad=k == 1) for k in range(3)]
    b = rx.Batch(reqs)
    b.run(rx.FP64)
    b.sync()
    (y0, s0), (y1, s1), (y2, s2) = (b.output(i) for i in range(3))
    b.close()
    assert s0 == 0 and s2 == 0 and s1 != 0
    assert np.all(y1 == 0) and np.any(y0 > 0) and conv_err(y2, y0) < 1e-8
    y, s = rx.eval_model(model, reqs[1]["params"], e, reqs[1].get("flux_in"), raise_on_error=False)
    assert s == s1 and np.all(y == 0)
