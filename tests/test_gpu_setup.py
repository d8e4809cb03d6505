"""k_setup at the edges of its tiles against the oracle: fine grids of one chunk,
around the workgroup sizes and the largest, tables whose axes are longer than a
wavefront (brackets in several loads a lane), the lamp post's reflection
fractions, and batches with the wide and the narrow workgroups.

Tolerance: 1e-8, the FP64 bar of the parity tests (the profile's sums are FP64 in
another order); 1e-12 between two workgroup sizes."""
import numpy as np
import pytest

import oracle
import relxill_amd as rx
from tests.helpers import RELLINE_CFG0, draw_lp_params, log_grid, rel_err, tables

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[(3, 2, 5, 2, 2, 3), (70, 66, 256, 130, 66, 256), (25, 22, 100, 20, 100, 100)])
def tabs(request):
    n_a, n_mu0, n_r, l_a, l_h, l_r = request.param
    rx.tables_synthetic(1, n_a, n_mu0, n_r, 8)
    rx.lptable_synthetic(3, l_a, l_h, l_r)
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    rel, lp = rx.tables_view()
    yield oracle.Tables(rel, lp)
    rx.tables_synthetic(1, 25, 22, 100, 20)
    rx.lptable_synthetic(3, 20, 100, 100)
    assert rx.lib.rx_init(0) == 0


@pytest.mark.parametrize("nr_fine", [64, 65, 511, 512, 513, 1000, 4096])
def test_fine_grids_and_table_axes(tabs, nr_fine):
    e = log_grid(400, 0.1, 10.0)
    assert rx.lib.rx_set_nr_fine(nr_fine) == 0
    try:
        cases = [(rx.MODEL_RELLINE, oracle.MOD_RELLINE, RELLINE_CFG0)]
        cases += [(rx.MODEL_RELLINELP, oracle.MOD_RELLINELP, p) for p in draw_lp_params(3, seed=nr_fine)]
        for model, omodel, p in cases:
            rp, st = oracle.rel_params(omodel, p)
            ref, _, st2 = oracle.relbase(tabs, rp, e / p[0], nr_fine=nr_fine)
            b = rx.Batch([dict(model=model, energy=e, params=p)])
            b.run(rx.FP64)
            b.sync()
            y, st_g = b.output(0)
            refl = b.reflfrac(0) if model == rx.MODEL_RELLINELP else None
            b.close()
            assert st == 0 and (st_g == 0) == (st2 == 0), (p, st2, st_g)
            if st2 == 0:
                assert rel_err(y, ref) < 1e-8
                if refl is not None:
                    want = oracle.system_parameters(tabs, rp, nr_fine=nr_fine)[0]["refl"]
                    np.testing.assert_allclose(refl, want, rtol=1e-10)
    finally:
        rx.lib.rx_set_nr_fine(1000)


def test_workgroup_sizes_agree():
    tables()
    assert rx.lib.rx_init(0) == 0
    e = log_grid(60, 1.0, 9.0)
    ps = draw_lp_params(257, seed=8)
    outs = []
    for n in (256, 257):  # wide and narrow workgroups
        b = rx.Batch([dict(model=rx.MODEL_RELLINELP, energy=e, params=p) for p in ps[:n]])
        b.run(rx.FP64)
        b.sync()
        outs.append([b.output(i)[0] for i in range(256)])
        b.close()
    assert max(rel_err(x, y) for x, y in zip(*outs)) < 1e-12
