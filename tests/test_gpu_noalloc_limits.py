"""The allocation-free entry point on grids whose work list of short segments does
not fit its scratch memory (it takes longer ones), beside sizes that fit: against
rx_eval_model.  Line models add radius chunks in any order: 1e-12 with margin."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import log_grid, rel_err, tables
from tests.test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr_fine,n", [(1000, 16384), (4096, 9000), (4096, 12000), (4096, 20000)])
def test_fine_grids(nr_fine, n):
    tables()
    try:
        assert rx.lib.rx_set_nr_fine(nr_fine) == 0
        assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
        e = log_grid(n, 0.1, 10.0)
        p = rx.DEFAULTS[rx.MODEL_RELLINE]
        y, st = _noalloc(rx.MODEL_RELLINE, p, e, None, rx.FP64)
        ref, st1 = rx.eval_model(rx.MODEL_RELLINE, p, e)
        assert st == 0 and st1 == 0 and np.any(ref > 0)
        assert rel_err(y, ref) < 1e-12
    finally:
        rx.lib.rx_set_nr_fine(1000)
        assert rx.lib.rx_init(0) == 0
