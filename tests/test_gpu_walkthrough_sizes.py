"""The walkthrough's two all-pairs passes over the sizes where their split
changes: fewer spheres than a workgroup owns, a partner round that ends
inside, at and past the last sphere, and both sides of each size rule.

Tolerances (normwise, infinity norm, vs FP64) as test_gpu_rpy.py: force, U
and Omega 1e-5, positions 1e-6."""
import ctypes as C

import numpy as np
import pytest

import orc
import sphx

pytestmark = pytest.mark.gpu


def near_field(pos):
    """Kern_getForce (:257-300) in FP64."""
    x = pos.astype(np.float64)
    out = np.zeros_like(x)
    for i0 in range(0, len(x), 512):
        d = x[None] - x[i0:i0 + 512, None]
        r = np.linalg.norm(d, axis=-1)
        k = np.arange(len(d))
        r[k, i0 + k] = np.inf
        i, j = np.nonzero(r < 1.5)
        fac = 5 * (np.exp(1.5 / r[i, j]) - 2.7128 * r[i, j] / 1.5)
        np.add.at(out, i0 + i, -d[i, j] * fac[:, None])
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 5, 255, 256, 257, 1024, 1025, 8192, 8195])
@pytest.mark.parametrize("with_force", [0, 1])
def test_walkthrough_sizes(gpu, n, with_force):
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3)))
    place = rng.permutation(m ** 3)[:n]
    pos = np.stack([place % m, place // m % m, place // (m * m)], 1) * 1.9
    pos = (pos + rng.uniform(-0.4, 0.4, (n, 3))).astype(np.float32)
    f0 = rng.normal(0, 1, (n, 3)).astype(np.float32)
    disp = np.zeros(n, sphx.display_dtype)
    disp["pos"], disp["type"] = pos, 7
    print(f"walkthrough n={n} force={with_force}", flush=True)
    # U and Omega start as garbage: without a node grid the background is zero
    arr = [sphx.DeviceArray(np.full((n, 3), np.nan, np.float32)), sphx.DeviceArray(disp),
           sphx.DeviceArray(np.full((n, 3), np.nan, np.float32)), sphx.DeviceArray(f0)]
    buf = sphx.StokesianBufList(*[a.ptr.value for a in arr], 0.01, 1.0)
    sphx.check(sphx.lib().sphx_rpy_walkthrough(None, C.byref(buf), n, with_force), "walkthrough")
    u, d, w, f = (a.get() for a in arr)
    ref = f0 + near_field(pos) if with_force else f0
    assert orc.relerr(f, ref) <= 1e-5
    ur, wr, pr = orc.rpy_walkthrough(pos, f, np.zeros((n, 3)), 0.01)
    assert orc.relerr(u, ur) <= 1e-5
    assert orc.relerr(d["pos"], pr) <= 1e-6
    if n > 1:
        assert orc.relerr(w, wr) <= 1e-5
    else:
        assert not w.any()
    np.testing.assert_array_equal(d["type"], 7)
