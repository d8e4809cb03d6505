"""k_rrad's two forms (a workgroup per incident zone for up to 24 requests, one per
four zones beyond): the same request by itself and in a batch of 25, for tables of
odd numbers of energy-shift bins and the most radial zones, line and relxill models.

The sums over the energy-shift bins are taken in another order (at most 20 FP64
terms of one sign): 1e-12 for lines with margin; convolved spectra the suite's
1e-8 (conv_err)."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import conv_err, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rad,n_g", [(50, 20), (64, 7), (9, 1), (33, 5)])
def test_forms(n_rad, n_g):
    tables()
    rx.xilltable_synthetic(5, 4, 3, 4, 3, 10, 300)
    rx.rradtable_synthetic(7, 21, n_rad, n_g)
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    try:
        e = log_grid(400, 0.2, 50.0)
        # h beta a Incl Rin Rout z gamma logxi Afe Ecut refl_frac returnrad boost
        lp = [4.0, 0.0, 0.97, 35.0, -1.0, 400.0, 0.0, 2.1, 2.7, 1.5, 120.0, 1.0, 1.0, 0.0]
        line = list(rx.DEFAULTS[rx.MODEL_RELLINELP])
        line[9] = 1.0  # return_rad
        for model, p in ((rx.MODEL_RELXILLLP, lp), (rx.MODEL_RELLINELP, line)):
            req = dict(model=model, energy=e, params=p)
            ys = []
            for n in (1, 25):
                b = rx.Batch([req] * n)
                b.run(rx.FP64)
                b.sync()
                y, st = b.output(n - 1)
                b.close()
                assert st == 0 and np.any(y > 0)
                ys.append(y)
            if model == rx.MODEL_RELLINELP:
                assert rel_err(ys[1], ys[0]) < 1e-12
            else:
                assert conv_err(ys[1], ys[0]) < 1e-8
    finally:
        rx.rradtable_synthetic(7, 21, 50, 20)
        rx.xilltable_synthetic()
        assert rx.lib.rx_init(0) == 0


@pytest.mark.parametrize("others", [False, True])
def test_solves_beside_sums(others):
    """k_before_rrad: relxilllpCp's solves beside the band sums (up to 32 requests)
    and before them (33), with and without other models in the batch."""
    tables()
    rx.xilltable_synthetic(5, 4, 3, 4, 3, 10, 300)
    rx.xillcptable_synthetic(6, 4, 3, 4, 3, 10, 300)
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    try:
        e = log_grid(300, 0.2, 50.0)
        cp = list(rx.DEFAULTS[rx.MODEL_RELXILLLPCP])
        lp = [4.0, 0.0, 0.97, 35.0, -1.0, 400.0, 0.0, 2.1, 2.7, 1.5, 120.0, 1.0, 1.0, 0.0]
        first = [dict(model=rx.MODEL_RELXILLLPCP, energy=e, params=cp)]
        if others:
            first += [dict(model=rx.MODEL_RELXILLLP, energy=e, params=lp),
                      dict(model=rx.MODEL_XILLVER, energy=e, params=rx.DEFAULTS[rx.MODEL_XILLVER]),
                      dict(model=rx.MODEL_RELXILL, energy=e, params=rx.DEFAULTS[rx.MODEL_RELXILL])]
        few, many = rx.Batch(first), rx.Batch(first + [first[0]] * 33)
        for b in (few, many):
            b.run(rx.FP64)
            b.sync()
        for i in range(len(first)):
            (y, st), (ref, st1) = many.output(i), few.output(i)
            assert st == 0 and st1 == 0 and np.any(ref > 0)
            assert conv_err(y, ref) < 1e-8
        np.testing.assert_array_equal(many.zones(0, 10), few.zones(0, 10))
        few.close()
        many.close()
    finally:
        rx.xilltable_synthetic()
        rx.xillcptable_synthetic()
        assert rx.lib.rx_init(0) == 0
