"""The RPY apply's default reduction segments are 16 a row tile at every size
(an FP32 sum of n/16 spheres per partial): above 4,096 spheres too the default
gives the bits of 16 segments set by hand, and its error against a dense FP64
product on sampled rows stays within the mode's bound (test_gpu_rpy.py's)."""
import numpy as np
import pytest

import orc
import sphx
from test_gpu_rpy_direct import BOUND, spheres

pytestmark = pytest.mark.gpu


def sampled(pos, rad, mu, F, rows):
    x, a = pos.astype(np.float64), rad.astype(np.float64)
    U = np.zeros((3 * len(rows), F.shape[1]))
    G = F.astype(np.float64).reshape(len(x), 3, -1)
    for t, i in enumerate(rows):
        d = x - x[i]
        r2 = (d ** 2).sum(1)
        r2[i] = 1
        c = 1 / (8 * np.pi * mu * np.sqrt(r2))
        s2 = (a[i] ** 2 + a ** 2) / r2
        c1, c2 = c * (1 + s2 / 3), c * (1 - s2) / r2
        c1[i], c2[i] = 1 / (6 * np.pi * mu * a[i]), 0
        dot = np.einsum("na,nak->nk", d, G) * c2[:, None]
        U[3 * t:3 * t + 3] = np.einsum("n,nak->ak", c1, G) + np.einsum("na,nk->ak", d, dot)
    return U


@pytest.mark.parametrize("mode", [1, 3, 6])
@pytest.mark.parametrize("n, K", [(320, 64), (700, 48), (1100, 32), (2049, 16), (4096, 64), (8192, 16),
                                  (16385, 16)])
def test_default_segments_lose_nothing(gpu, n, K, mode):
    pos, rad, r = spheres(n, n)
    F = r.standard_normal((3 * n, K)).astype(np.float32)
    rows = r.permutation(n)[:200]
    ref = sampled(pos, rad, 1.3, F, rows)
    at = (3 * rows[:, None] + np.arange(3)).ravel()
    with sphx.Mobility(n, K) as m:
        m.set_spheres(pos, rad, 1.3)
        U = m.apply(F, mode)
        m.set_split(16)
        V = m.apply(F, mode)
    rms = lambda x: np.sqrt(np.mean((x[at] - ref) ** 2) / np.mean(ref ** 2))
    print(f"n={n} K={K} mode={mode}: default {rms(U):.3e} / {orc.relerr(U[at], ref):.3e}, "
          f"16 segments {rms(V):.3e} / {orc.relerr(V[at], ref):.3e}", flush=True)
    np.testing.assert_array_equal(U, V)
    assert orc.relerr(U[at], ref) <= BOUND[mode]
