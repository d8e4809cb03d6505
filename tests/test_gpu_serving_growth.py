"""Servers whose slots grow: bursts of growing and shrinking size, from one small
request to more than a pinned request block and a slot's first memory hold, at a
server with room and at one whose budget is less than a slot's first memory, equal
batches of the same requests.

Tolerance: a burst is cut into batches as slots come free, and other segments and
forms add the same values in another order (1e-12; conv_err at 1e-8 for the
convolutions, 1e-13 of the maximum)."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import conv_err, draw_lp_params, draw_relconv_params, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


def _requests(n):
    sizes = np.exp(np.random.default_rng(3).uniform(np.log(50), np.log(9000), n)).astype(int)
    lp, cv = draw_lp_params(n, seed=1), draw_relconv_params(n, seed=2)
    out = []
    for k, nb in enumerate(sizes):
        if k % 2:
            out.append(dict(model=rx.MODEL_RELLINELP, energy=log_grid(int(nb), 0.1, 10.0), params=lp[k]))
        else:
            e = log_grid(int(nb), 0.1, 100.0)
            out.append(dict(model=rx.MODEL_RELCONV, energy=e, params=cv[k], flux_in=e[:-1] ** -2.0 * np.diff(e)))
    return out


@pytest.mark.parametrize("budget", [16 << 30, 3 << 20])
@pytest.mark.parametrize("prec", [0, 1])
def test_growing_bursts(budget, prec):
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    reqs = _requests(300)
    b = rx.Batch(reqs)
    b.run(prec)
    b.sync()
    ref = [b.output(i)[0] for i in range(len(reqs))]
    b.close()
    srv = rx.Server(max_inflight=4096, hbm_budget=budget, n_streams=3, precision=prec)
    try:
        for n in (1, 3, 40, 300, 2, 300, 40):
            tickets = srv.replay(reqs[:n], np.zeros(n))
            srv.drain()
            for i, t in enumerate(tickets):
                y, st, _ = srv.poll(t)
                assert st == 0
                assert (conv_err(y, ref[i]) < 1e-8) if i % 2 == 0 else (rel_err(y, ref[i]) < 1e-12)
    finally:
        srv.stop()
