"""The RPY apply where its route is chosen by size: one launch in FP32 for few
spheres, the tile path otherwise, and the tile path for a caller who set its
split or whose arrays are not 16-byte aligned or are the same, against a dense
FP64 product.

Tolerances (normwise, infinity norm) as test_gpu_rpy.py: the direct route
holds every mode to mode 6's 1e-5; the tile path 1e-5, 1e-4 and 2e-2."""
import ctypes as C

import numpy as np
import pytest

import orc
import sphx

pytestmark = pytest.mark.gpu
BOUND = {1: 2e-2, 3: 1e-4, 6: 1e-5}


def spheres(n, seed):
    r = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    place = r.permutation(m ** 3)[:n]
    pos = np.stack([place % m, place // m % m, place // (m * m)], 1) * 0.125
    pos = (pos + r.uniform(-0.03, 0.03, (n, 3))).astype(np.float32)
    return pos, r.uniform(0.01, 0.03, n).astype(np.float32), r


def dense(pos, rad, mu, F):
    x, a = pos.astype(np.float64), rad.astype(np.float64)
    U = np.zeros(F.shape)
    for i in range(len(x)):
        d = x - x[i]
        r2 = (d ** 2).sum(1)
        r2[i] = 1
        c = 1 / (8 * np.pi * mu * np.sqrt(r2))
        s2 = (a[i] ** 2 + a ** 2) / r2
        M = (c * (1 + s2 / 3))[:, None, None] * np.eye(3) + (c * (1 - s2) / r2)[:, None, None] * d[:, :, None] * d[:, None, :]
        M[i] = np.eye(3) / (6 * np.pi * mu * a[i])
        U[3 * i:3 * i + 3] = M.transpose(1, 0, 2).reshape(3, -1) @ F.astype(np.float64)
    return U


# both sides of each size rule, and edges of the workgroup's spheres and threads
@pytest.mark.parametrize("n, K, direct", [(1, 16, 1), (2, 64, 1), (3, 32, 1), (255, 48, 1), (256, 16, 1),
                                          (257, 64, 1), (306, 64, 1), (307, 64, 0), (1024, 16, 1),
                                          (1025, 16, 0), (512, 32, 1), (513, 32, 0), (512, 48, 1), (513, 48, 0)])
@pytest.mark.parametrize("mode", [1, 3, 6])
def test_routes(gpu, n, K, direct, mode):
    pos, rad, r = spheres(n, n)
    F = r.standard_normal((3 * n, K)).astype(np.float32)
    ref = dense(pos, rad, 1.3, F)
    print(f"rpy n={n} K={K} mode={mode}", flush=True)
    with sphx.Mobility(n, K) as m:
        m.set_spheres(pos, rad, 1.3)
        e = orc.relerr(m.apply(F, mode), ref)
        print(f"  {e:.2e}")
        assert e <= (1e-5 if direct else BOUND[mode])
        # an input 4 bytes past a 16-byte boundary
        pad = sphx.DeviceArray(np.concatenate([np.zeros(1, np.float32), F.ravel()]))
        out = sphx.DeviceArray(np.full((3 * n, K), np.nan, np.float32))
        m.apply_device(pad.ptr.value + 4, out.ptr.value, mode)
        m.sync()
        assert orc.relerr(out.get(), ref) <= BOUND[mode]
        # in place
        both = sphx.DeviceArray(F)
        m.apply_device(both.ptr.value, both.ptr.value, mode)
        m.sync()
        assert orc.relerr(both.get(), ref) <= BOUND[mode]
        # the tile path with a split of the caller's
        m.set_split(3)
        assert orc.relerr(m.apply(F, mode), ref) <= BOUND[mode]
