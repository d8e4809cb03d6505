"""k_primary's split of the caller bins over workgroups: every split gives the
bits of the one-bin-a-thread split, for grids of one bin, of one workgroup's
bins, one less, one more, and for batches whose threads take several bins.

The xillver models have no sums whose order could change, so their outputs are
equal to the bit; relxill's profile adds the radius chunks in any order (FP64),
a few 1e-16 of a bin per addition: 1e-12 with margin."""
import numpy as np
import pytest

import relxill_amd as rx
from tests.helpers import conv_err, log_grid, tables

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def small_tables():
    tables()
    assert rx.lib.rx_init(0) == 0, rx.lib.rx_last_error()
    rx.xilltable_synthetic(5, 4, 3, 4, 3, 5, 300)
    rx.xillcptable_synthetic(6, 4, 3, 4, 3, 5, 300)
    yield
    rx.xilltable_synthetic()
    rx.xillcptable_synthetic()


@pytest.mark.parametrize("n_bins,n_req", [(1, 3), (255, 5), (256, 5), (257, 1100), (513, 1100), (1300, 700)])
@pytest.mark.parametrize("model", [rx.MODEL_XILLVER, rx.MODEL_XILLVERCP, rx.MODEL_RELXILL])
def test_split_over_workgroups(small_tables, n_bins, n_req, model):
    e = log_grid(n_bins, 0.3, 60.0)
    rng = np.random.default_rng(n_bins)
    ps = []
    for _ in range(n_req):
        p = list(rx.DEFAULTS[model])
        p[8 if model == rx.MODEL_RELXILL else 0] = rng.uniform(1.4, 2.6)
        ps.append(p)
    b = rx.Batch([dict(model=model, energy=e, params=p) for p in ps])
    b.run(rx.FP64)
    b.sync()
    for i in (0, n_req // 2, n_req - 1):
        (y, st), (ref, st1) = b.output(i), rx.eval_model(model, ps[i], e)
        assert st == 0 and st1 == 0 and np.all(ref > 0)
        if model == rx.MODEL_RELXILL:
            assert conv_err(y, ref) < 1e-12
        else:
            np.testing.assert_array_equal(y, ref)
    b.close()
