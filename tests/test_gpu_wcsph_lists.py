"""The WCSPH density and force passes' neighbour lists: every route of the
two passes (few and many lanes per particle, short and long lists, lists
that overflow to the cell scan, cell rows too long for a list entry, keys
older than the positions, no list at all) against the oracle on identical
inputs.

Tolerances as test_gpu_sph.py: normwise against the FP64 oracle, 1e-5 for
the density and 1e-4 for pressure and force, or 4x the CPU-FP32
restatement's own error (the sums' order differs)."""
import numpy as np
import pytest

import sphx
from helpers import assert_close, options, shuffled_scene, state_from_gpu

pytestmark = pytest.mark.gpu


def scene(n, family, cluster=0, h=0.02, seed=11):
    L = (0.01 * (n[0] + 6), 0.01 * (n[1] + 4), 0.01 * n[2])
    p, disp, calc, _ = shuffled_scene(*n, L=L, h=h, seed=seed, kernel_family=family,
                                      n_out=min(5, n[0] * n[1] * n[2] // 8))
    rng = np.random.default_rng(seed)
    fluid = np.where(disp["type"] == 0)[0]
    calc["vel"][fluid] = rng.normal(0, 0.05, (len(fluid), 3))
    calc["visc"][fluid] = 1e-3
    if cluster:
        # many particles inside one support: lists (and, past 4096 in a row
        # of cells, their entries) overflow
        at = np.array([0.035, 0.035, 0.035])
        disp["pos"][fluid[:cluster]] = at + rng.uniform(-0.004, 0.004, (cluster, 3))
    o = options(wcsph_kernel=family)
    if family == 1:
        o.eos_B = 1000.0 * 20.0 ** 2 / 7.0
        o.art_visc_alpha, o.sound_speed = 0.01, 20.0
    return p, disp, calc, o


def check(ctx, p, o, force_first=False):
    def both(kernel):
        s = [state_from_gpu(ctx, p, t, o, iisph=False) for t in (np.float32, np.float64)]
        for x in s:
            getattr(x, kernel)()
        return s

    if not force_first:
        s32, s64 = both("density_pressure")
        ctx.call("wcsph_density_pressure")
        _, c = ctx.download()
        m = (s32["type"] != 1) & (s32["mgcell"] != 0xFFFFFFFF)
        assert_close("1/rho", c["dens"], s32["dens"], s64["dens"], 1e-5, m)
        assert_close("pressure", c["pressure"], s32["pressure"], s64["pressure"], 1e-4, m)
    s32, s64 = both("force")
    ctx.call("wcsph_force")
    _, c = ctx.download()
    m = (s32["type"] != 1) & (s32["mgcell"] != 0xFFFFFFFF)
    assert_close("accel", c["accel"], s32["accel"], s64["accel"], 1e-4, m)


@pytest.mark.parametrize("family", [0, 1])
@pytest.mark.parametrize("n, cluster", [((1, 1, 1), 0), ((5, 3, 2), 0), ((9, 8, 7), 0),
                                        ((9, 8, 7), 450), ((18, 17, 17), 4700), ((33, 31, 32), 0)])
def test_density_and_force_routes(gpu, family, n, cluster):
    p, disp, calc, o = scene(n, family, cluster)
    print(f"lists family={family} n={len(disp)} cluster={cluster}", flush=True)
    with sphx.Context(p, o) as ctx:
        ctx.upload(disp, calc)
        ctx.call("grid_build")
        ctx.call("boundary_volume")
        check(ctx, p, o)


@pytest.mark.parametrize("family", [0, 1])
def test_keys_older_than_the_positions(gpu, family):
    """Passes called after an advance without a new grid scan the 27 cells
    of the old keys, as the reference's would."""
    p, disp, calc, o = scene((10, 9, 8), family)
    p.dt = 2e-2   # moves particles by up to some tenths of a cell
    with sphx.Context(p, o) as ctx:
        ctx.upload(disp, calc)
        ctx.call("grid_build")
        ctx.call("boundary_volume")
        ctx.call("wcsph_density_pressure")
        ctx.call("wcsph_advance")
        check(ctx, p, o)


def test_force_without_a_list_of_this_support(gpu):
    """The force pass builds its own list when the density pass has not run
    for these positions, or ran with the other kernel family's support."""
    p, disp, calc, o = scene((9, 8, 7), 1)
    with sphx.Context(p, o) as ctx:
        ctx.upload(disp, calc)
        ctx.call("grid_build")
        ctx.call("boundary_volume")
        ctx.call("wcsph_density_pressure")
        o.wcsph_kernel = 0
        ctx.set_options(o)
        check(ctx, p, o, force_first=True)
        ctx.call("grid_build")
        check(ctx, p, o, force_first=True)
