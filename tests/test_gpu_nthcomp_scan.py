"""The nthcomp solve's scans (a run of rows per lane) at the ends of the
accepted parameters, where a lane has few rows, many rows or none at the end of
the grid, and the bracket of an edge at and beyond both ends of the photon
grid, against the oracle's row-by-row elimination.

Tolerance: 1e-10 of a bin as in the other nthcomp tests (the elimination's own
round-off is a few 1e-14 a point), bins below 1e-12 of the largest E F_E
relative to that."""
import numpy as np
import pytest

import oracle
import relxill_amd as rx
from tests.helpers import log_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kte", [0.1, 0.35, 1.0, 17.0, 400.0, 1e4])
@pytest.mark.parametrize("gam", [1.01, 1.7, 3.4, 9.9])
def test_solve_and_brackets(kte, gam):
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    for lo, hi, n in ((1e-7, 1e6, 777), (4e-6, 6e-6, 50), (0.1, 100.0, 300)):
        e = log_grid(n, lo, hi)
        y = rx.nthcomp(e, kte, gam, 0.7)[0]
        ref = oracle.nthcomp(e, kte, gam, 0.7)
        ok = np.isfinite(ref)
        np.testing.assert_array_equal(np.isfinite(y), ok)
        # E F_E of a bin: photons times E^2 / dE
        w = (0.5 * (e[1:] + e[:-1])) ** 2 / np.diff(e)
        scale = np.abs(ref * w)[ok].max() if ok.any() else 0.0
        err = np.max(np.abs(y - ref)[ok] * w[ok] / np.maximum(np.abs(ref * w)[ok], 1e-12 * scale)) if scale > 0 else 0.0
        print(f"nthcomp kTe {kte} Gamma {gam} [{lo}, {hi}]: {err:.2e}", flush=True)
        assert err < 1e-10
