"""k_conv's workgroups: the wide form (up to 256 units in a run) against the
narrow one, on the smallest and largest convolution grids and those around the
widest workgroup.

The transforms' arithmetic does not depend on the width; the block sums are taken
in another order (at most 8192 positive FP64 terms) and the profile's radius
chunks add in any order: 1e-12 with margin (the spectra stay within a factor 100
of their maximum)."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import conv_err, log_grid, tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [256, 512, 1024, 4096, 8192])
def test_width(n):
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    e = log_grid(301, 0.2, 80.0)
    rng = np.random.default_rng(n)
    spec = e[:-1] ** -1.2 * np.diff(e) * (1 + 0.3 * np.sin(5 * np.log(e[:-1])))
    ps = []
    for _ in range(257):
        p = list(rx.DEFAULTS[rx.MODEL_RELCONV])
        p[3], p[4] = rng.uniform(-0.9, 0.99), rng.uniform(15, 80)
        ps.append(p)
    try:
        assert rx.lib.rx_set_conv_grid(n, 0.00035, 2000.0) == 0
        b = rx.Batch([dict(model=rx.MODEL_RELCONV, energy=e, params=p, flux_in=spec) for p in ps])
        b.run(rx.FP64)
        b.sync()
        for i in (0, 128, 256):
            (y, st), (one, st1) = b.output(i), rx.eval_model(rx.MODEL_RELCONV, ps[i], e, spec)
            assert st == 0 and st1 == 0
            assert conv_err(y, one) < 1e-12
        b.close()
    finally:
        assert rx.lib.rx_set_conv_grid(4096, 0.00035, 2000.0) == 0
