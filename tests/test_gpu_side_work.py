"""Distributions, zone records and primaries that go with another kernel's launch
(few requests) against the same as launches of their own (more than 8192 windows,
more than 256 requests with a primary), for batches of one model and mixed ones.

Zone records are computed by the same code from the same values: equal bits.  The
distributions add chunks in any order: at most 16 x 10 FP64 terms, 1e-13 with
margin.  Spectra: the convolutions of faint bins, the suite's 1e-8."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import conv_err, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def small_tables():
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    rx.xilltable_synthetic(5, 4, 3, 4, 3, 10, 300)
    rx.xillcptable_synthetic(6, 4, 3, 4, 3, 10, 300)
    yield
    rx.xilltable_synthetic()
    rx.xillcptable_synthetic()


def request(model, e, rng):
    p = list(rx.DEFAULTS[model])
    if model == rx.MODEL_RELXILLLP:
        p[1] = rng.uniform(-0.9, 0.9)
    elif model == rx.MODEL_RELXILL:
        p[4] = rng.uniform(20, 70)
    return dict(model=model, energy=e, params=p)


@pytest.mark.parametrize("precision", [rx.FP64, rx.FP32])
@pytest.mark.parametrize("models", [(rx.MODEL_RELXILL,), (rx.MODEL_RELXILLLP,),
                                    (rx.MODEL_RELXILL, rx.MODEL_XILLVER, rx.MODEL_RELLINE, rx.MODEL_RELXILLLP)])
def test_alone_and_in_a_large_batch(small_tables, models, precision):
    rng = np.random.default_rng(len(models))
    e = log_grid(90, 0.3, 60.0)
    reqs = [request(models[k % len(models)], e, rng) for k in range(1040)]
    big = rx.Batch(reqs)
    big.run(precision)
    big.sync()
    for i in (0, 1, 2, 3, 519, 1038, 1039):
        one = rx.Batch([reqs[i]])
        one.run(precision)
        one.sync()
        (y, st), (ref, st1) = big.output(i), one.output(0)
        assert st == 0 and st1 == 0 and np.any(ref > 0)
        assert conv_err(y, ref) < 1e-8
        nz = {rx.MODEL_RELXILL: 1, rx.MODEL_RELXILLLP: 10}.get(reqs[i]["model"], 0)
        if nz:
            np.testing.assert_array_equal(big.zones(i, nz), one.zones(0, nz))
            assert rel_err(big.dist(i, 10 * nz), one.dist(0, 10 * nz)) < 1e-13
        one.close()
    big.close()
