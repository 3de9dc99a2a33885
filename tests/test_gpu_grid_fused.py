"""sphx_grid_build folds its stages into fewer launches; its results against
hash, sort and reorder called one by one, bit for bit: keys, order, ranges,
the born-id table, particles, fractions and MPM state, over one to three
radix passes (an odd count starts in the other buffer) and both ways of
summing the tiles' histograms (up to 200 tiles of 2,048 keys, and more)."""
import numpy as np
import pytest

import sphx

pytestmark = pytest.mark.gpu


def build(p, disp, calc, alpha, rounds, stages):
    out = []
    with sphx.Context(p) as c:
        c.upload(disp, calc)
        c.mf_setup([1000.0, 1.2], [1e-6, 1.5e-5])
        c.mf_upload(alpha)
        c.mpm_setup(1, 1)
        for r in range(rounds):
            for s in stages:
                c.call(s)
            d, q = c.download()
            out.append((d, q, c.download_grid(), c.mf_download()))
            # move some particles (by id, the same in both) for the next round
            rng = np.random.default_rng(r)
            step = rng.normal(0, 0.05, (len(d), 3)).astype(np.float32)
            d["pos"] += np.where(rng.random(len(d)) < 0.3, 1, 0)[q["bornid"], None] * step[q["bornid"]]
            f = out[-1][3]["alpha"]
            c.upload(d, q)
            c.mf_upload(f)
    return out


@pytest.mark.parametrize("n, res", [(1, 8), (70, 8), (2047, 16), (2049, 64), (5000, 256),
                                    (196608, 64), (196609, 64), (300000, 256)])
def test_fused_build_equals_stages(gpu, n, res):
    p, disp, calc, _ = sphx.scene_sand(n=n, lo=0.0, hi=1.0, dx=1.0 / res, res=res, seed=n)
    rng = np.random.default_rng(n)
    order = rng.permutation(n)
    disp, calc = disp[order].copy(), calc[order].copy()
    calc["bornid"] = np.arange(n)
    calc["stress"] = rng.normal(0, 1, (n, 9))
    calc["B"] = rng.normal(0, 1, (n, 9))
    alpha = rng.uniform(0, 1, (n, 2)).astype(np.float32)
    out = rng.random(n) < 0.02   # out of the grid
    disp["pos"][out] = -7.0
    print(f"build n={n} res={res}", flush=True)
    a = build(p, disp, calc, alpha, 2, ["grid_build"])
    b = build(p, disp, calc, alpha, 2, ["grid_hash", "grid_sort", "grid_reorder"])
    for (d, q, g, m), (d2, q2, g2, m2) in zip(a, b):
        np.testing.assert_array_equal(d, d2)
        np.testing.assert_array_equal(q, q2)
        for k in g:
            np.testing.assert_array_equal(g[k], g2[k], err_msg=k)
        for k in m:
            np.testing.assert_array_equal(m[k], m2[k], err_msg=k)
    # and the first round against a stable sort
    g = a[0][2]
    ref = np.argsort(np.where(g["mgcell"] == 0xFFFFFFFF, np.uint32(p.gridtotal), g["mgcell"]), kind="stable")
    np.testing.assert_array_equal(ref, np.arange(n))
    key = np.empty(n, np.int64)
    key[g["midsort"]] = np.where(g["mgcell"] == 0xFFFFFFFF, p.gridtotal, g["mgcell"])
    np.testing.assert_array_equal(g["midsort"], np.argsort(key, kind="stable"))


@pytest.mark.parametrize("n, res", [(409600, 64), (409601, 64), (409600, 256), (409601, 256)])
def test_both_ways_of_summing_the_histograms(gpu, n, res):
    test_fused_build_equals_stages(gpu, n, res)
