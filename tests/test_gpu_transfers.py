"""Transfers that are packed on the device: uploads and downloads of whole
contexts, of ranges, in several chunks of the staging ring and after a
reorder, and the fractions', bit for bit against what went in."""
import numpy as np
import pytest

import sphx

pytestmark = pytest.mark.gpu


def particles(n, seed):
    """Every field of both packs filled with its own random bits (finite)."""
    r = np.random.default_rng(seed)
    disp, calc = np.zeros(n, sphx.display_dtype), np.zeros(n, sphx.calc_dtype)
    for a in (disp, calc):
        for f in a.dtype.names:
            a[f] = r.uniform(0.1, 1.0, a[f].shape)
    disp["type"] = r.integers(0, 2, n) | r.integers(0, 3, n) << 8
    calc["bornid"] = np.arange(n)
    return disp, calc


def context(cap):
    p, _, _, _ = sphx.scene_dambreak(4, 4, 4)
    p.num, p.maxNum = 0, cap
    return sphx.Context(p)


# one particle; a wave's and a workgroup's edges; the ring's slot edges
# (9,362 packs of 224 bytes in 2 MiB) and more chunks than slots
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 9362, 9363, 50001])
def test_round_trip(gpu, n):
    disp, calc = particles(n, n)
    with context(n + 5) as c:
        c.upload(disp, calc)
        d, q = c.download()
        np.testing.assert_array_equal(d, disp)
        np.testing.assert_array_equal(q, calc)
        # a range in the middle, replaced and read back alone
        a, b = n // 3, n // 3 + (n + 2) // 3
        d2, q2 = particles(b - a, n + 1)
        q2["bornid"] = calc["bornid"][a:b]
        c.upload(d2, q2, start=a)
        disp[a:b], calc[a:b] = d2, q2
        L = sphx.lib()
        dr, qr = np.zeros(b - a, sphx.display_dtype), np.zeros(b - a, sphx.calc_dtype)
        sphx.check(L.sphx_download(c.h, sphx.ptr(dr), sphx.ptr(qr), a, b - a))
        np.testing.assert_array_equal(dr, disp[a:b])
        np.testing.assert_array_equal(qr, calc[a:b])
        # appended after a reorder, then replaced as a whole
        c.call("grid_build")
        d1, q1 = c.download()
        da, qa = particles(5, n + 2)
        c.upload(da, qa, start=n)
        d, q = c.download()
        np.testing.assert_array_equal(d, np.concatenate([d1, da]))
        np.testing.assert_array_equal(q, np.concatenate([q1, qa]))
        c.call("grid_build")
        d3, q3 = particles(n + 5, n + 3)
        c.upload(d3, q3)
        only = np.zeros(n + 5, sphx.display_dtype)
        sphx.check(L.sphx_download(c.h, sphx.ptr(only), None, 0, n + 5))
        np.testing.assert_array_equal(only, d3)
        np.testing.assert_array_equal(c.download()[1], q3)


@pytest.mark.parametrize("nphase", [1, 2, 3])
@pytest.mark.parametrize("n", [1, 300, 200001])
def test_fractions_round_trip(gpu, n, nphase):
    disp, calc = particles(n, 7)
    r = np.random.default_rng(n)
    alpha = r.uniform(0, 1, (n, nphase)).astype(np.float32)
    rho, nu = np.float32([1000.0, 1.2, 700.0][:nphase]), np.float32([1e-6, 1.5e-5, 3e-6][:nphase])
    with context(n) as c:
        c.upload(disp, calc)
        c.mf_setup(rho, nu)
        a = n // 4
        c.mf_upload(alpha[:a])
        c.mf_upload(alpha[a:], start=a)
        out = c.mf_download()
        rm, nm = np.zeros(n, np.float32), np.zeros(n, np.float32)
        for k in range(nphase):
            rm = rm + alpha[:, k] * rho[k]
            nm = nm + alpha[:, k] * nu[k]
        np.testing.assert_array_equal(out["alpha"], alpha)
        np.testing.assert_array_equal(out["rho_m"], rm)
        g = np.float32(c.params.gravity.tolist())
        np.testing.assert_array_equal(out["mforce"], np.broadcast_to(g, (n, 3)))
        np.testing.assert_array_equal(out["drift"], 0)
        _, q = c.download()
        fluid = (disp["type"] & 0xFF) != 1
        np.testing.assert_array_equal(q["visc"], np.where(fluid, nm, calc["visc"]))
