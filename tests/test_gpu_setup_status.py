"""The status of a request whose lamp post's reflection fraction is refused
(photons to infinity and to the disk above all photons) while its fine radii are
evaluated beside it: the same in every evaluation, in both widths of k_setup's
workgroups, with zero flux, and the neighbours of such a request unharmed."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import draw_lp_params, log_grid, tables

pytestmark = pytest.mark.gpu


@pytest.fixture
def odd_table(tmp_path):
    """the synthetic lamp-post table, emission angles of 0 inside 100 rg and pi outside"""
    tables()
    path = str(tmp_path / "lp.rxtb").encode()
    assert rx.lib.rx_lptable_save(path) == 0
    raw = np.fromfile(path.decode(), dtype=np.float32)
    n_a, n_h, n_r = raw[:5].view(np.int32)[2:]
    o_rad = 5 + n_a + n_a * n_h
    o_del = o_rad + n_a * n_r + n_a * n_h * n_r
    rad = raw[o_rad:o_rad + n_a * n_r].reshape(n_a, 1, n_r)
    d = raw[o_del:o_del + n_a * n_h * n_r].reshape(n_a, n_h, n_r)
    d[:] = np.where(rad > 100.0, np.pi, 0.0)
    d[:, :, -1] = 0.0
    raw.tofile(path.decode())
    assert rx.lib.rx_lptable_load(path) == 0, rx.lib.rx_last_error()
    assert rx.lib.rx_init(0) == 0
    yield
    rx.lptable_synthetic(3, 20, 100, 100)
    assert rx.lib.rx_init(0) == 0


def test_reflection_status(odd_table):
    e = log_grid(300, 0.1, 10.0)
    par = draw_lp_params(1, seed=2)[0]
    for _ in range(20):
        y, st = rx.eval_model(rx.MODEL_RELLINELP, par, e, raise_on_error=False)
        assert st != 0 and not y.any()
        assert b"status 20" in rx.lib.rx_last_error()
    line = list(rx.DEFAULTS[rx.MODEL_RELLINE])
    ref, st = rx.eval_model(rx.MODEL_RELLINE, line, e)
    assert st == 0
    for n in (8, 300):
        b = rx.Batch([dict(model=rx.MODEL_RELLINELP, energy=e, params=par),
                      dict(model=rx.MODEL_RELLINE, energy=e, params=line)] * (n // 2))
        b.run(rx.FP64)
        b.sync()
        for i in range(n):
            y, st = b.output(i)
            assert (st == 0) == (i % 2 == 1)
            np.testing.assert_allclose(y, ref if i % 2 else 0 * ref, rtol=1e-10, atol=1e-12 * ref.max())
        b.close()
