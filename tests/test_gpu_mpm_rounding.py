"""The MPM stencil's weights round as the reference's quotient by the node
spacing does, also for a spacing that is no power of two: root mean square
errors of P2G's node masses, the stress pass's densities and G2P's velocities
against the FP64 oracle, next to the FP32 oracle's, which performs the same
operations (bound as test_gpu_wcsph_edges.py's: a tenth above it)."""
import numpy as np
import pytest

import sphx
from test_gpu_mpm import oracle_from

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("res, n", [(23, 3000), (47, 40000)])
def test_errors_are_the_fp32_oracles(gpu, kernel, res, n):
    p, disp, calc, _ = sphx.scene_sand(n=n, lo=0.2, hi=0.7, dx=1.0 / res, res=res, seed=n)
    rng = np.random.default_rng(n)
    calc["vel"] = rng.normal(0, 0.3, (n, 3))
    calc["B"] = rng.normal(0, 0.01, (n, 9))
    calc["stress"] = rng.normal(0, 400, (n, 9))

    def twins(ctx, nodes=True):
        return [oracle_from(ctx, p, kernel, kernel, nodes, t) for t in (np.float64, np.float32)]

    def compare(name, gpu_val, ref, f32):
        e, e32 = (np.sqrt(np.mean((np.asarray(x, np.float64) - ref) ** 2)) for x in (gpu_val, f32))
        print(f"{name}: {e:.3e}, FP32 oracle {e32:.3e}", flush=True)
        assert e <= 1.1 * e32

    with sphx.Context(p) as ctx:
        ctx.upload(disp, calc)
        ctx.mpm_setup(kernel, kernel)
        ctx.call("grid_build")
        (_, a), (_, b) = twins(ctx, nodes=False)
        a.p2g(1), b.p2g(1), ctx.mpm_p2g(1)
        compare("node mass", ctx.mpm_nodes()[1], a["node_m"], b["node_m"])
        (s, a), (t, b) = twins(ctx)
        a.stress(), b.stress(), ctx.call("mpm_stress")
        compare("density", ctx.download()[1]["dens"], s["dens"], t["dens"])
        (s, a), (t, b) = twins(ctx)
        a.g2p(1), b.g2p(1), ctx.mpm_g2p(1)
        compare("velocity", ctx.download()[1]["vel"], s["vel"], t["vel"])
