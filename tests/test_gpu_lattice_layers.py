"""The lattice product where a wave marches two layers (2048 waves or more: long
boxes here, so that few points are enough), with an even and an odd number of
layers (the last chunk whole or half) and planes that do not fill their waves:
CG iterates with it against CG on the assembled matrix, from a right side that
loads every point."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# waves = ceil(points of a plane / 62) ceil(layers / 2); points 12, 65, 62 and
# 63; below the line one layer per wave: the same mesh a few layers shorter.  The
# last two: waves so empty that the element-wise product is the faster one, and
# the same nearly so
@pytest.mark.parametrize("mesh", [(3, 2, 4099), (2, 3, 4100), (12, 4, 2047), (30, 1, 4096), (20, 2, 2046), (3, 2, 4089),
                                  (1, 1, 16000), (1, 1, 8000)])
def test_two_layers_per_wave(mastg, mesh):
    nx, ny, nz = mesh
    print(f"[lattice layers] {mesh}", flush=True)
    k, j, i = np.meshgrid(np.arange(nz + 1), np.arange(ny + 1), np.arange(nx + 1), indexing="ij")
    xyz = np.stack([i.ravel() * 1.0, j.ravel() * 1.25, k.ravel() * 0.75], -1)
    corner = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
    c, b, a = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    conn = np.stack([(a + p + (nx + 1) * (b + q + (ny + 1) * (c + r))).ravel() for p, q, r in corner], -1).astype(np.int32)
    rng = np.random.default_rng(5)
    nodes = rng.choice(len(xyz), len(xyz) // 10, replace=False)      # constraints anywhere
    con = np.sort(nodes * 6 + rng.integers(0, 3, len(nodes)))
    desc = mastg.desc_from_arrays(mastg.HEX8_ELASTIC, xyz, conn, 6, constrained_dofs=con, E=72e9, nu=0.33, penalty=3.0)
    ctx = mastg.Context(desc)
    ctx._keep = desc
    ctx.set_params(rng.uniform(0.3, 1.0, len(conn)))
    ctx.assemble()
    rhs = rng.standard_normal(ctx.n_dofs)
    rhs[con] = 0.0
    # the product to 1e-12 of its largest value, as everywhere; a few
    # well-conditioned steps add a factor of ten at most
    for n in (1, 2, 6):
        opts = dict(rtol=1e-14, max_iters=n, raise_on_error=False)
        x, _ = ctx.solve(rhs, solver=mastg.SOLVER_CG_JACOBI, **opts)
        y, st = ctx.solve(rhs, solver=mastg.SOLVER_MATFREE, **opts)
        assert st["iters"] == n and np.abs(x).max() > 0
        assert np.max(np.abs(x - y)) <= 1e-11 * np.abs(x).max()
    ctx.close()
