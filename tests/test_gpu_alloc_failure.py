"""An allocation that the device refuses (far more than it has) is reported by the
call that asked for it, and by no later one."""
import ctypes

import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import RELLINE_CFG0, log_grid, tables

pytestmark = pytest.mark.gpu
RX_ERR_NOMEM = 102


def test_refused_allocation():
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    e = log_grid(500, 0.1, 10.0)
    ref, st = rx.eval_model(rx.MODEL_RELLINE, RELLINE_CFG0, e)
    assert st == 0
    for _ in range(2):
        ms = ctypes.c_double(0.0)
        assert rx.lib.rx_copy_test(1 << 45, 1, ctypes.byref(ms)) == RX_ERR_NOMEM
        y, st = rx.eval_model(rx.MODEL_RELLINE, RELLINE_CFG0, e)
        assert st == 0
        np.testing.assert_allclose(y, ref, rtol=1e-10, atol=1e-12 * ref.max())
