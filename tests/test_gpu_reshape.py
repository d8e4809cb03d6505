"""Work shapes set between a run and the reading of its results: outputs,
statuses, angle distributions, zone records and reflection fractions are the
run's, whatever the new shape's work list takes, and the next run's are equal
to them.

Tolerances: what is read again is the same bits.  Two shapes of one batch add
the same values in another order (1e-12); a ten-zone convolution carries a
round-off of 1e-13 of its maximum (conv_err at 1e-8)."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import conv_err, draw_lp_params, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


def _read(b, n):
    out = [b.output(i) for i in range(n)]
    return ([y for y, _ in out], [st for _, st in out], [rx.lib.rx_batch_status(b.h, i) for i in range(n)],
            [b.reflfrac(i) for i in range(n)], b.dist(0, 10), b.zones(0, 10))


@pytest.fixture(scope="module")
def dev():
    tables()
    rx.xilltable_synthetic(5, 4, 3, 4, 3, 10, 600)
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    yield
    rx.xilltable_synthetic()


@pytest.mark.parametrize("shapes", [[(1, 0)], [(4096, 0), (1, 8), (3, 0)]])
@pytest.mark.parametrize("prec", [0, 1])
def test_results_outlive_a_shape(dev, prec, shapes):
    e = log_grid(2000, 0.1, 100.0)
    reqs = [dict(model=rx.MODEL_RELXILLLP, energy=e, params=list(rx.DEFAULTS[rx.MODEL_RELXILLLP]))]
    for p in draw_lp_params(12, seed=4):
        reqs.append(dict(model=rx.MODEL_RELLINELP, energy=e, params=p))
    bad = list(reqs[-1]["params"])
    bad[4], bad[5] = 400.0, 20.0  # Rin beyond Rout: refused
    reqs.append(dict(model=rx.MODEL_RELLINELP, energy=e, params=bad))
    n = len(reqs)
    b = rx.Batch(reqs)
    try:
        b.set_shape(256, 0)
        b.run(prec)
        b.sync()
        ref = _read(b, n)
        assert ref[1][:-1] == [0] * (n - 1) and ref[1][-1] != 0
        for shape in shapes:
            b.set_shape(*shape)
            got = _read(b, n)
            assert got[1] == ref[1] and got[2] == ref[2]
            for k in (0, 3):
                for x, y in zip(got[k], ref[k]):
                    np.testing.assert_array_equal(x, y)
            np.testing.assert_array_equal(got[4], ref[4])
            np.testing.assert_array_equal(got[5], ref[5])
        b.run(prec)
        b.sync()
        new = _read(b, n)[0]
        assert conv_err(new[0], ref[0][0]) < 1e-8
        for x, y in zip(new[1:], ref[0][1:]):
            assert rel_err(x, y) < 1e-12
    finally:
        b.close()
