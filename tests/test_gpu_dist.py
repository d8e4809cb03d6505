"""The emission-angle distribution (k_dist) at the edges of its tiles against
the oracle: fine grids of one chunk, of a chunk and one radius and of the
default size, tables of few and of the most g* points (several rounds of
staged node rows) and few and many angle bins.

Tolerance: the sums hold at most 1000 x 128 positive FP64 terms in another
order than the oracle's, 1.3e5 x 1.1e-16 = 1.4e-11 at worst."""
import numpy as np
import pytest

import oracle
import relxill_amd as rx
from tests.helpers import log_grid, reflection_spectrum, rel_err

pytestmark = pytest.mark.gpu

TOL = 1.4e-11


@pytest.mark.parametrize("n_g", [3, 20, 64])
@pytest.mark.parametrize("nr_fine", [64, 65, 1000])
@pytest.mark.parametrize("n_incl", [1, 10, 64])
def test_distribution_tiles(n_g, nr_fine, n_incl):
    rx.tables_synthetic(1, 6, 5, 100, n_g)
    e_ref, refl = reflection_spectrum(n_bins=400, n_incl=n_incl)
    e_out = log_grid(300, 0.1, 100.0)
    try:
        assert rx.lib.rx_set_nr_fine(nr_fine) == 0
        assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
        rel, lp = rx.tables_view()
        T = oracle.Tables(rel, lp)
        cg = log_grid(4096, 0.00035, 2000.0)
        sid = rx.reflset_create(e_ref, refl)
        for p in ([3.0, 3.0, 15.0, 0.9, 30.0, -1.0, 400.0, 0.0], [4.0, 2.0, 9.0, -0.5, 75.0, 12.0, 900.0, 0.0]):
            _, ref, st = oracle.relxill_conv(T, p, cg, e_ref, refl, e_out, nr_fine=nr_fine)
            b = rx.Batch([dict(model=rx.MODEL_RELXILL_CONV, energy=e_out, params=p, refl_set=sid)])
            b.run(rx.FP64)
            b.sync()
            d, st_g = b.dist(0, n_incl), b.output(0)[1]
            b.close()
            assert st == 0 and st_g == 0
            err = rel_err(d, ref)
            print(f"dist n_g {n_g} nr {nr_fine} n_incl {n_incl}: {err:.2e}", flush=True)
            assert err < TOL
    finally:
        rx.lib.rx_reflsets_clear()
        rx.lib.rx_set_nr_fine(1000)
        rx.tables_synthetic(1, 25, 22, 100, 20)
        np.testing.assert_equal(rx.lib.rx_init(0), 0)
