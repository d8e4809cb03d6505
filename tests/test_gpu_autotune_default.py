"""The autotuner never settles for less than the default: a batch of one request,
whose default segments of one or two bins its other candidates (32 bins and more)
cannot match, keeps them, and the calls of its class with it."""
import pytest

import relxill_amd as rx
from tests.helpers import RELLINE_CFG0, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
def test_short_segments_kept(prec):
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    e = log_grid(777, 0.1, 10.0)  # (a class of its own among the tests: the choice stays)
    ref, st = rx.eval_model(rx.MODEL_RELLINE, RELLINE_CFG0, e, precision=prec)
    b = rx.Batch([dict(model=rx.MODEL_RELLINE, energy=e, params=RELLINE_CFG0)])
    try:
        seg, _ = b.autotune(prec)
        assert seg < 32
        b.run(prec)
        b.sync()
        y, st2 = b.output(0)
    finally:
        b.close()
    z, st3 = rx.eval_model(rx.MODEL_RELLINE, RELLINE_CFG0, e, precision=prec)
    assert st == st2 == st3 == 0
    assert rel_err(y, ref) < 1e-12 and rel_err(z, ref) < 1e-12
