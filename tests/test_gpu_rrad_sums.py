"""The zones' returning-radiation correction factors (k_zone, k_before_rrad,
k_rrad) at the edges of their tiles against the oracle: xillver tables of one
workgroup's bins, one less, one more and several workgroups, 4 and 10
inclinations (those of 2, 3 or 5 give the synthetic tables a negative average and status 41), a table whose band 0.15-500 keV reaches beyond its last edge when
shifted, a density division (logN off 15) and an ionisation gradient.

Tolerance: conv_err's 1e-8, the bar of the relxilllp tests (relative down to
1e-5 of the maximum; the factors themselves are FP64 sums)."""
import pytest

import oracle
import relxill_amd as rx
from tests.helpers import conv_err, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu

TOL = 1e-8


@pytest.fixture(scope="module")
def tabs():
    _, _, T = tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    yield T
    rx.xilltable_synthetic()
    rx.xillcptable_synthetic()


@pytest.mark.parametrize("n_incl", [4, 10])
@pytest.mark.parametrize("n_ener", [255, 256, 257, 1100])
def test_correction_factors(tabs, n_ener, n_incl):
    T = tabs
    e = log_grid(500, 0.1, 100.0)
    rx.xilltable_synthetic(5, 5, 3, 4, 5, n_incl, n_ener)
    rx.xillcptable_synthetic(6, 5, 3, 4, 5, n_incl, n_ener)
    xa, xc = oracle.Xill(rx.xilltable_view()), oracle.Xill(rx.xilltable_view(nthcomp=True))
    # h beta a Incl Rin Rout z gamma logxi Afe Ecut refl_frac returnrad boost
    cases = [(rx.MODEL_RELXILLLP, oracle.MOD_RELXILLLP, xa,
              [h, 0.0, a, 35.0, -1.0, rout, 0.0, 2.1, 2.7, 1.5, ec, 1.0, 1.0, 0.0])
             for h, a, rout, ec in ((3.0, 0.998, 400.0, 120.0), (30.0, 0.5, 900.0, 20.0))]
    # Incl a Rin Rout h beta gamma logxi logN Afe kTe refl_frac z iongrad_index iongrad_type returnrad boost
    cases += [(rx.MODEL_RELXILLLPCP, oracle.MOD_RELXILLLPCP, xc,
               [35.0, 0.9, -1.0, 400.0, 5.0, 0.0, 2.1, 2.7, dens, 1.5, 40.0, 1.0, 0.0, 1.3, grad, 1.0, 0.0])
              for dens, grad in ((15.0, 0.0), (17.3, 0.0), (16.0, 1.0))]
    for model, omodel, xt, p in cases:
        ref, dref, st = oracle.relxill_model(omodel, T, xt, p, e)
        b = rx.Batch([dict(model=model, energy=e, params=p)])
        b.run(rx.FP64)
        b.sync()
        (y, st_g), d = b.output(0), b.dist(0, dref.size)
        b.close()
        assert st == 0 and st_g == 0, p
        err, derr = conv_err(y, ref), rel_err(d, dref.reshape(-1))
        print(f"rrad sums {n_ener} {n_incl} {p}: {err:.2e} dist {derr:.2e}", flush=True)
        assert err < TOL and derr < TOL
