"""Transfers through staging memory of other sizes than the default (the
smallest is the route of a context for which memory is short), changed between
transfers of one context: bit for bit what went in."""
import numpy as np
import pytest

import sphx
from helpers import options
from test_gpu_transfers import context, particles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 18, 19, 72, 73, 3000, 20000])
def test_round_trip_at_each_size(gpu, n):
    """18 packs of 224 bytes fill a slot of 4 KiB, 72 the four slots."""
    disp, calc = particles(n, n)
    alpha = np.random.default_rng(n).uniform(0, 1, (n, 3)).astype(np.float32)
    with context(n) as c:
        for kib in (1, 16, 100, 0, 4096, 16, 1 << 20):
            c.set_options(options(staging_kib=kib))
            c.upload(disp, calc)
            d, q = c.download()
            np.testing.assert_array_equal(d, disp)
            np.testing.assert_array_equal(q, calc)
            c.call("grid_build")
            g = c.download_grid()
            assert sorted(g["midsort"]) == list(range(n))
            c.mf_setup([1000.0, 800.0, 1.2], [1e-6, 1e-6, 1.5e-5])
            c.mf_upload(alpha)
            np.testing.assert_array_equal(c.mf_download()["alpha"], alpha)
            d, q = c.download()   # after the reorder, as the default size gives it
            c.set_options(options())
            d0, q0 = c.download()
            np.testing.assert_array_equal(d, d0)
            np.testing.assert_array_equal(q, q0)
