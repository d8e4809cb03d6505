"""Convolutions of inputs of any size: the result is linear in the input's scale
over hundreds of decades, for the cut of the transforms that few units and that
many units take, with a renormalised profile and with a lamp post's.

Tolerance: scaled by a power of two an input goes through the same roundings, up
to the order in which the profile's radius chunks add: conv_err at 1e-8, that is
1e-13 of the maximum."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import conv_err, log_grid, tables

pytestmark = pytest.mark.gpu
EXPONENTS = [-660, -548, -300, -40, 1, 40, 300, 548, 660]


@pytest.fixture(scope="module")
def dev():
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()


def _input(e):
    return e[:-1] ** -1.2 * np.diff(e) * (1 + 0.3 * np.sin(5 * np.log(e[:-1])))


@pytest.mark.parametrize("model", [rx.MODEL_RELCONV, 12])  # 12: relconv_lp
@pytest.mark.parametrize("prec", [0, 1])
def test_few_units(dev, model, prec):
    e = log_grid(301, 0.2, 80.0)
    f, par = _input(e), list(rx.DEFAULTS[model])
    ref, st = rx.eval_model(model, par, e, f, precision=prec)
    assert st == 0
    for k in EXPONENTS:
        y, st = rx.eval_model(model, par, e, np.ldexp(f, k), precision=prec)
        assert st == 0 and conv_err(np.ldexp(y, -k), ref) < 1e-8, k


@pytest.mark.parametrize("model", [rx.MODEL_RELCONV, 12])
@pytest.mark.parametrize("prec", [0, 1])
def test_many_units(dev, model, prec):
    e = log_grid(301, 0.2, 80.0)
    f, par = _input(e), list(rx.DEFAULTS[model])
    ref, st = rx.eval_model(model, par, e, f, precision=prec)
    assert st == 0
    reqs = [dict(model=model, energy=e, params=par, flux_in=np.ldexp(f, EXPONENTS[i % len(EXPONENTS)]))
            for i in range(257)]
    b = rx.Batch(reqs)
    b.run(prec)
    b.sync()
    for i, k in enumerate(EXPONENTS):
        y, st = b.output(i)
        assert st == 0 and conv_err(np.ldexp(y, -k), ref) < 1e-8, k
    b.close()
