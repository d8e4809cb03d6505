"""Admission by the device working set: the work list of a small batch, whose
segments are short, counts in full.  One line request of 8000 bins takes about
0.4 MB and its list 0.5 MB: within 1.2 MB they run one at a time, within 16 MB
together."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import RELLINE_CFG0, log_grid, tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("budget,alone", [(1200 << 10, True), (16 << 20, False)])
def test_list_counts(budget, alone):
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    reqs = [dict(model=rx.MODEL_RELLINE, energy=log_grid(8000, 0.1, 10.0), params=RELLINE_CFG0)] * 40
    srv = rx.Server(max_inflight=64, hbm_budget=budget, n_streams=4, precision=rx.FP32)
    try:
        tickets = srv.replay(reqs, np.zeros(len(reqs)))
        srv.drain()
        assert all(srv.poll(t)[1] == 0 for t in tickets)
        stats = srv.stats()
    finally:
        srv.stop()
    if alone:
        assert stats["batches"] == len(reqs) and stats["max_concurrent_batches"] == 1, stats
    else:
        assert stats["batches"] < len(reqs), stats
