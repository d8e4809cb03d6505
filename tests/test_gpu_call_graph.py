"""Evaluation calls on one grid replay their launch graph while the line's energy
and the redshift vary, on grids that hold the whole line and on grids that cut it
at either end, and give what calls without graphs give.

Tolerance: the profile's radius chunks add in any order, and the segments differ
between the two (1e-12)."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import RELLINE_CFG0, draw_lp_params, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    yield
    rx.lib.rx_set_graphs(1)


@pytest.mark.parametrize("n_bins,lo,hi", [(1000, 2.0, 10.0), (300, 4.0, 9.0), (3000, 0.1, 10.0), (40, 5.0, 6.0)])
@pytest.mark.parametrize("model", [rx.MODEL_RELLINE, rx.MODEL_RELLINELP])
@pytest.mark.parametrize("prec", [0, 1])
def test_replays(dev, model, n_bins, lo, hi, prec):
    e = log_grid(n_bins, lo, hi)
    base = list(RELLINE_CFG0) if model == rx.MODEL_RELLINE else draw_lp_params(1, seed=6)[0]
    zi = 8 if model == rx.MODEL_RELLINE else 6
    pars = []
    for k in range(40):
        p = list(base)
        p[0], p[zi] = 6.4 + 0.02 * (k * 7 % 20), 0.002 * (k * 5 % 20)
        pars.append(p)
    rx.lib.rx_set_graphs(0)
    ref = [rx.eval_model(model, p, e, precision=prec)[0] for p in pars]
    rx.lib.rx_set_graphs(1)
    for p in pars[:8]:
        rx.eval_model(model, p, e, precision=prec)
    before = rx.lib.rx_call_graph_replays()
    for p, r in zip(pars, ref):
        y, st = rx.eval_model(model, p, e, precision=prec)
        assert st == 0 and rel_err(y, r) < 1e-12
    # (a call with a longer reach than any before it may widen the list once or twice)
    assert rx.lib.rx_call_graph_replays() - before >= 34
