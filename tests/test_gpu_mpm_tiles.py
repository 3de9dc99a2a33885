"""The MPM scatter's tiles at the sizes where their handling changes: one
particle, partial waves and workgroups, boxes around the tile's 2,048 nodes
(one LDS window on one side, several on the other) and past the 16,384 a
tile may have (straight to the nodes), boundary particles in between; P2G, stress, node force and G2P of both splines against the FP64
oracle with test_gpu_mpm.py's bounds."""
import numpy as np
import pytest

import sphx
from test_gpu_mpm import check, check_nodes, oracle_from, sand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("n, cells", [(1, 1), (63, 3), (256, 5), (257, 5), (700, 9), (256, 10),
                                      (256, 11), (512, 12), (900, 16), (300, 22),
                                      (300, 27)])
def test_tile_sizes(gpu, kernel, n, cells):
    lo = 0.3 if cells < 27 else 0.08
    p, disp, calc = sand(kernel, kernel, n=n, lo=lo, hi=lo + cells / 32, seed=n + cells)
    if n > 10:
        disp["type"][5::7] = sphx.TYPE_BOUNDARY
    print(f"tiles kernel={kernel} n={n} cells={cells}", flush=True)
    with sphx.Context(p) as ctx:
        ctx.upload(disp, calc)
        ctx.mpm_setup(kernel, kernel)
        ctx.call("grid_build")
        st, mp = oracle_from(ctx, p, kernel, kernel, nodes=False)
        mp.p2g(1)
        s32, m32 = oracle_from(ctx, p, kernel, kernel, nodes=False, dtype=np.float32)
        m32.p2g(1)
        ctx.mpm_p2g(1)
        v, m = ctx.mpm_nodes()
        check("p2g mass", m, mp["node_m"])
        check_nodes("p2g", v, m, mp["node_v"], mp["node_m"], m32["node_v"])
        st, mp = oracle_from(ctx, p, kernel, kernel)
        mp.stress()
        ctx.call("mpm_stress")
        d, c = ctx.download()
        fl = d["type"] != sphx.TYPE_BOUNDARY
        check("density", c["dens"][fl], st["dens"][fl])
        check("stress", c["stress"][fl], mp["stress"][fl])
        st, mp = oracle_from(ctx, p, kernel, kernel)
        mp.node_update()
        s32, m32 = oracle_from(ctx, p, kernel, kernel, dtype=np.float32)
        m32.node_update()
        ctx.call("mpm_node_update")
        v, m = ctx.mpm_nodes()
        check_nodes("node update", v, m, mp["node_v"], mp["node_m"], m32["node_v"])
        st, mp = oracle_from(ctx, p, kernel, kernel)
        mp.g2p(1)
        ctx.mpm_g2p(1)
        d, c = ctx.download()
        check("g2p velocity", c["vel"][fl], st["vel"][fl])
        check("g2p B", c["B"][fl], mp["B"][fl])


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("n", [65535, 65536, 65537])
def test_gather_lanes(gpu, kernel, n):
    """Stress and G2P on both sides of the size where four lanes stop sharing
    a particle."""
    p, disp, calc = sand(kernel, kernel, n=n, lo=0.2, hi=0.2 + 20 / 32, seed=n)
    disp["type"][5::7] = sphx.TYPE_BOUNDARY
    print(f"lanes kernel={kernel} n={n}", flush=True)
    with sphx.Context(p) as ctx:
        ctx.upload(disp, calc)
        ctx.mpm_setup(kernel, kernel)
        ctx.call("grid_build")
        ctx.mpm_p2g(1)
        st, mp = oracle_from(ctx, p, kernel, kernel)
        mp.stress()
        ctx.call("mpm_stress")
        d, c = ctx.download()
        fl = d["type"] != sphx.TYPE_BOUNDARY
        check("density", c["dens"][fl], st["dens"][fl])
        check("stress", c["stress"][fl], mp["stress"][fl])
        st, mp = oracle_from(ctx, p, kernel, kernel)
        mp.g2p(1)
        ctx.mpm_g2p(1)
        d, c = ctx.download()
        check("g2p velocity", c["vel"][fl], st["vel"][fl])
        check("g2p B", c["B"][fl], mp["B"][fl])
