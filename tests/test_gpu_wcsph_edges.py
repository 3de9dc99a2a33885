"""The WCSPH density and force passes where their lists' route could differ
from the plain loops over the 27 cells: densities, velocities and parameters
that a caller may set between the stages, and the rounding of a single pair,
against the oracle on identical inputs.

Tolerances of the scene tests as test_gpu_wcsph_lists.py.  The pair test's:
the FP32 oracle performs the same operations, each rounded correctly, on the
same inputs, and the GPU contracts some of them, so its mean error over a few
thousand independent pairs may not exceed the FP32 oracle's by more than a
tenth (sampling noise of the two means)."""
import numpy as np
import pytest

import sphx
from helpers import assert_close, options, shuffled_scene, state_from_gpu

pytestmark = pytest.mark.gpu


def scene(family, seed=5, n=(11, 9, 8)):
    L = tuple(0.01 * (m + 5) for m in n)
    p, disp, calc, _ = shuffled_scene(*n, L=L, h=0.02, seed=seed, kernel_family=family, n_out=4)
    rng = np.random.default_rng(seed)
    fluid = np.where(disp["type"] == 0)[0]
    calc["vel"][fluid] = rng.normal(0, 0.05, (len(fluid), 3))
    calc["visc"][fluid] = 1e-3
    o = options(wcsph_kernel=family)
    o.art_visc_alpha, o.sound_speed = 0.01, 20.0
    return p, disp, calc, o, rng, fluid


def force_matches(ctx, p, o):
    s32, s64 = (state_from_gpu(ctx, p, t, o, iisph=False) for t in (np.float32, np.float64))
    for s in (s32, s64):
        s.force()
    ctx.call("wcsph_force")
    _, c = ctx.download()
    m = (s32["type"] != 1) & (s32["mgcell"] != 0xFFFFFFFF)
    assert np.isfinite(s64["accel"][m]).all() and np.isfinite(c["accel"][m]).all()
    assert_close("accel", c["accel"], s32["accel"], s64["accel"], 1e-4, m)


def density_matches(ctx, p, o):
    s32, s64 = (state_from_gpu(ctx, p, t, o, iisph=False) for t in (np.float32, np.float64))
    for s in (s32, s64):
        s.density_pressure()
    ctx.call("wcsph_density_pressure")
    _, c = ctx.download()
    m = (s32["type"] != 1) & (s32["mgcell"] != 0xFFFFFFFF)
    assert_close("1/rho", c["dens"], s32["dens"], s64["dens"], 1e-5, m)
    assert_close("pressure", c["pressure"], s32["pressure"], s64["pressure"], 1e-4, m)


@pytest.mark.parametrize("family", [0, 1])
@pytest.mark.parametrize("zero", [1.0, 0.5])
def test_force_of_uploaded_densities(gpu, family, zero):
    """A force pass before any density pass uses the uploaded 1/rho, which
    the scene generators leave zero: finite, and the oracle's."""
    p, disp, calc, o, rng, fluid = scene(family)
    calc["dens"][fluid] = np.where(rng.random(len(fluid)) < zero, 0.0, 1e-3)
    calc["pressure"][fluid] = rng.uniform(0, 500, len(fluid))
    with sphx.Context(p, o) as ctx:
        ctx.upload(disp, calc)
        ctx.call("grid_build")
        ctx.call("boundary_volume")
        force_matches(ctx, p, o)


@pytest.mark.parametrize("family", [0, 1])
def test_boundary_velocities_stay_out_of_the_viscosity(gpu, family):
    """A wall particle adds friction only where the fluid approaches it; its
    velocity enters nothing else."""
    p, disp, calc, o, rng, fluid = scene(family)
    wall = np.where(disp["type"] == 1)[0]
    calc["vel"][rng.choice(wall, len(wall) // 2, replace=False)] = np.nan
    with sphx.Context(p, o) as ctx:
        ctx.upload(disp, calc)
        ctx.call("grid_build")
        ctx.call("boundary_volume")
        ctx.call("wcsph_density_pressure")
        force_matches(ctx, p, o)


@pytest.mark.parametrize("family", [0, 1])
@pytest.mark.parametrize("hashed", ["grid_hash", "grid_build"])
def test_grid_moved_between_hash_and_sort(gpu, family, hashed):
    """Keys of the old grid stay in use until the next hash; the passes then
    scan all 27 cells of them."""
    p, disp, calc, o, _, _ = scene(family)
    with sphx.Context(p, o) as ctx:
        ctx.upload(disp, calc)
        ctx.call("grid_build")
        ctx.call("boundary_volume")
        ctx.call("wcsph_density_pressure")
        ctx.call("wcsph_force")
        ctx.call(hashed)
        cell = 1.0 / p.gridIdfac.x
        p.gridmin.x -= 0.45 * cell
        p.gridmin.y += 0.5 * cell
        p.gridmin.z -= 0.55 * cell
        ctx.set_params(p)
        ctx.call("grid_sort")
        if hashed == "grid_hash":
            ctx.call("grid_reorder")
        density_matches(ctx, p, o)
        force_matches(ctx, p, o)


@pytest.mark.parametrize("family", [0, 1])
@pytest.mark.parametrize("other", [0, 1])
def test_rounding_of_one_pair(gpu, family, other):
    """Pairs out of each other's reach, of two fluid particles or a fluid and
    a wall particle."""
    p, disp, calc, _ = sphx.scene_dambreak(17, 17, 17, 0.01, (1.4, 1.4, 1.4), 0.02, 2, 1e-4, 5, family)
    m = disp["type"] == 0
    disp, calc = disp[m].copy(), calc[m].copy()
    n = len(disp) // 2
    disp, calc = disp[:2 * n], calc[:2 * n]
    p.num = p.maxNum = 2 * n
    rng = np.random.default_rng(17 + family)
    at = np.stack(np.meshgrid(*[np.arange(14)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] * 0.095 + 0.05
    d = rng.normal(0, 1, (n, 3))
    d *= (rng.uniform(0.15, 0.95, n) * (0.04 if family else 0.02) / np.linalg.norm(d, axis=1))[:, None]
    disp["pos"][:n], disp["pos"][n:] = at, at + d
    disp["type"][n:] = other
    calc["vel"] = rng.normal(0, 0.5, (2 * n, 3))
    calc["visc"] = rng.uniform(1e-3, 2e-3, 2 * n)
    calc["dens"] = rng.uniform(0.9e-3, 1.1e-3, 2 * n)
    calc["pressure"] = rng.uniform(100, 500, 2 * n)
    calc["bornid"] = np.arange(2 * n)
    o = options(wcsph_kernel=family)
    o.art_visc_alpha, o.sound_speed = 0.3, 20.0
    with sphx.Context(p, o) as ctx:
        ctx.upload(disp, calc)
        ctx.call("grid_build")
        for kernel, field in (("force", "accel"), ("density_pressure", "dens")):
            s32, s64 = (state_from_gpu(ctx, p, t, o, iisph=False) for t in (np.float32, np.float64))
            for s in (s32, s64):
                getattr(s, kernel)()
            ctx.call("wcsph_" + kernel)
            _, c = ctx.download()
            fl = s32["type"] == 0
            assert fl.sum() >= n and (s32["mgcell"] != 0xFFFFFFFF).all()

            def mean_error(x):
                x, r = (np.asarray(a, np.float64)[fl].reshape(fl.sum(), -1) for a in (x, s64[field]))
                return np.mean(np.linalg.norm(x - r, axis=1) / np.linalg.norm(r, axis=1))

            e, e32 = mean_error(c[field]), mean_error(s32[field])
            print(f"{kernel}: mean error of a pair {e:.3e}, FP32 oracle {e32:.3e}", flush=True)
            assert e <= 1.1 * e32


@pytest.mark.parametrize("family", [0, 1])
@pytest.mark.parametrize("most", [-1, 8, 24, 0])
def test_lists_that_are_limited(gpu, family, most):
    """No list at all (as where its memory is short), lists that many or all
    particles overflow, and the limit lifted again: the same results."""
    p, disp, calc, o, _, _ = scene(family)
    o.wcsph_list_max = most
    with sphx.Context(p, o) as ctx:
        ctx.upload(disp, calc)
        ctx.call("grid_build")
        ctx.call("boundary_volume")
        density_matches(ctx, p, o)
        force_matches(ctx, p, o)
        o.wcsph_list_max = -1 if most == 0 else 0
        ctx.set_options(o)
        force_matches(ctx, p, o)
        density_matches(ctx, p, o)
        force_matches(ctx, p, o)


@pytest.mark.parametrize("family", [0, 1])
@pytest.mark.parametrize("n", [12288, 12289, 49152, 49153])
def test_both_sides_of_the_force_pass_sizes(gpu, family, n):
    """Counts at which the force pass changes the lanes that share a particle."""
    p, disp, calc, _ = sphx.scene_dambreak(37, 37, 37, 0.01, (0.37, 0.37, 0.37), 0.02, 2, 1e-4, n, family)
    fluid = np.where(disp["type"] == 0)[0][:n]
    disp, calc = disp[fluid].copy(), calc[fluid].copy()
    p.num = p.maxNum = n
    rng = np.random.default_rng(n)
    calc["vel"] = rng.normal(0, 0.05, (n, 3))
    calc["visc"] = 1e-3
    calc["bornid"] = np.arange(n)
    o = options(wcsph_kernel=family)
    o.art_visc_alpha, o.sound_speed = 0.01, 20.0
    with sphx.Context(p, o) as ctx:
        ctx.upload(disp, calc)
        ctx.call("grid_build")
        density_matches(ctx, p, o)
        force_matches(ctx, p, o)
