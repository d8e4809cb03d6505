"""How requests reach the device and results the host: outputs of one run read
in any order, several times, by several threads and across the read-ahead
windows are the same bits, and a new run's outputs are not the last run's; a
call whose request block or output is larger than the pinned memory equals the
batch's output; a call after calls of other sizes; rejected requests."""
import threading

import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import RELLINE_CFG0, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()


def _requests(sizes, gam0=2.0):
    out = []
    for k, n in enumerate(sizes):
        p = list(rx.DEFAULTS[rx.MODEL_XILLVER])
        p[0] = gam0 + 0.001 * k
        out.append(dict(model=rx.MODEL_XILLVER, energy=log_grid(n, 0.2, 90.0), params=p))
    return out


@pytest.mark.parametrize("sizes", [[1], [5, 3, 16384, 7], [16384] * 9, [300, 9000, 40000, 20] * 9, [700000, 11, 300000]])
def test_outputs_in_any_order(dev, sizes):
    b = rx.Batch(_requests(sizes))
    n = len(sizes)
    try:
        b.run(rx.FP64)
        seq = [b.output(i)[0] for i in range(n)]  # (waits for the run by itself)
        rng = np.random.default_rng(n)
        orders = [range(n), range(n - 1, -1, -1), rng.integers(0, n, 3 * n), list(range(n)) * 2, range(0, n, 2)]
        for order in orders:
            for i in order:
                y, st = b.output(int(i))
                assert st == 0
                np.testing.assert_array_equal(y, seq[int(i)])
        for i in (0, n - 1):
            ref, st = rx.eval_model(rx.MODEL_XILLVER, _requests(sizes)[i]["params"], log_grid(sizes[i], 0.2, 90.0))
            assert st == 0
            np.testing.assert_array_equal(ref, seq[i])
        b.run(rx.FP64)  # the windows of the run before are void
        b.sync()
        for i in range(n):
            np.testing.assert_array_equal(b.output(i)[0], seq[i])
        bad = []

        def read(part):
            for i in range(part, n, 3):
                if not np.array_equal(b.output(i)[0], seq[i]):
                    bad.append(i)

        ts = [threading.Thread(target=read, args=(k,)) for k in range(3)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not bad
    finally:
        b.close()


def test_reads_follow_the_last_run(dev):
    """FP32 and FP64 runs of one batch differ in their bits: what is read is the
    last run's."""
    e = log_grid(3000, 0.1, 10.0)
    b = rx.Batch([dict(model=rx.MODEL_RELLINE, energy=e, params=RELLINE_CFG0)] * 3)
    try:
        got = []
        for prec in (rx.FP64, rx.FP32, rx.FP64, rx.FP32):
            b.run(prec)
            b.sync()
            got.append([b.output(i)[0] for i in (0, 1, 2)])
        for k in (0, 1, 2):
            assert rel_err(got[2][k], got[0][k]) < 1e-12 and rel_err(got[3][k], got[1][k]) < 1e-12
            assert rel_err(got[1][k], got[0][k]) > 1e-9
    finally:
        b.close()


@pytest.mark.parametrize("sizes", [[3, 600000, 5, 200], [500000, 1, 530000, 64]])
def test_calls_of_any_size(dev, sizes):
    for n in sizes:
        e = log_grid(n, 0.3, 9.0)
        b = rx.Batch([dict(model=rx.MODEL_RELLINE, energy=e, params=RELLINE_CFG0)])
        b.run(rx.FP32)
        b.sync()
        ref, st = b.output(0)
        b.close()
        y, st1 = rx.eval_model(rx.MODEL_RELLINE, RELLINE_CFG0, e, precision=rx.FP32)
        assert st == 0 and st1 == 0 and rel_err(y, ref) < 1e-12
        bad = list(RELLINE_CFG0)
        bad[6], bad[7] = 50.0, 40.0
        y, st = rx.eval_model(rx.MODEL_RELLINE, bad, e, precision=rx.FP32, raise_on_error=False)
        assert st == rx.RX_ERR_PARAM and np.all(y == 0)
