"""Jacobian values into device memory from every row-assembly kernel: over the row
plan, by class without it (MASTG_OPT_ROW_ASSEMBLY 2) and from each cell's own
geometry, for rows of up to 27 blocks and of more than 42 (eight cells that share
one node and nothing else: 57).  Bitwise the host call's values, nothing around
them touched, and the element scatter's to 1e-12."""
import ctypes as C

import numpy as np
import pytest

from helpers import rel_err_floor

pytestmark = pytest.mark.gpu

CORNER = np.array([(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)])


def _box(mesh):
    nx, ny, nz = mesh
    k, j, i = np.meshgrid(np.arange(nz + 1), np.arange(ny + 1), np.arange(nx + 1), indexing="ij")
    xyz = np.stack([i.ravel(), j.ravel(), k.ravel()], -1).astype(float)
    e = np.array([(a, b, c) for c in range(nz) for b in range(ny) for a in range(nx)])
    p = e[:, None, :] + CORNER[None]
    return xyz, (p[..., 0] + (nx + 1) * (p[..., 1] + (ny + 1) * p[..., 2])).astype(np.int32)


def _pinwheel():
    """The eight unit cubes around the origin, joined at the origin alone."""
    xyz, conn = [np.zeros(3)], []
    for o in range(8):
        low = np.array([(o >> d & 1) - 1.0 for d in range(3)])
        cell = []
        for c in CORNER:
            x = low + c
            if x.any():
                cell.append(len(xyz))
                xyz.append(x)
            else:
                cell.append(0)
        conn.append(cell)
    return np.array(xyz), np.array(conn, np.int32)


@pytest.mark.parametrize("option", [1, 2])
@pytest.mark.parametrize("shape", ["one class", "two classes", "distorted"])
@pytest.mark.parametrize("mesh", ["box", "pinwheel"])
def test_device_values_of_every_row_kernel(mastg, mesh, shape, option):
    print(f"[row assembly, device J] {mesh}, {shape}, option {option}", flush=True)
    xyz, conn = _box((7, 5, 3)) if mesh == "box" else _pinwheel()
    if shape == "two classes":          # cells beyond a plane are longer
        xyz[:, 0] = np.where(xyz[:, 0] > (3 if mesh == "box" else 0), 1.5 * xyz[:, 0] - (1.5 if mesh == "box" else 0.0),
                             xyz[:, 0])
    elif shape == "distorted":
        xyz = xyz + np.random.default_rng(1).uniform(-0.08, 0.08, xyz.shape)
    desc = mastg.desc_from_arrays(mastg.HEX8_ELASTIC, xyz, conn, 6, constrained_dofs=np.array([6, 7, 8, 13, 20]),
                                  E=72e9, nu=0.33, penalty=3.0)
    ctx = mastg.Context(desc)
    ctx._keep = desc
    ctx.set_params(np.random.default_rng(2).uniform(0.2, 1.0, len(conn)))
    x = np.random.default_rng(3).standard_normal(ctx.n_dofs)
    ctx.set_option(mastg.OPT_ROW_ASSEMBLY, 0)
    R0, J0 = ctx.assemble(x)
    rp, _ = ctx.csr_pattern()
    assert (np.diff(rp).max() > 3 * 42) == (mesh == "pinwheel")
    ctx.set_option(mastg.OPT_ROW_ASSEMBLY, option)
    R, J = ctx.assemble(x)
    assert rel_err_floor(J, J0, rp, floor=1e-2) <= 1e-12
    assert np.max(np.abs(R - R0)) <= 1e-12 * np.abs(R0).max()
    host = np.full(J.nbytes + 32, 0x5A, np.uint8)
    L, dp, dx = mastg.lib(), C.c_void_p(), C.c_void_p()
    D = C.POINTER(C.c_double)
    ctx._chk(L.mastg_device_alloc(ctx.h, host.nbytes, C.byref(dp)))
    ctx._chk(L.mastg_device_alloc(ctx.h, x.nbytes, C.byref(dx)))
    try:
        ctx._chk(L.mastg_copy(ctx.h, dp, host.ctypes.data, host.nbytes, 0))
        ctx._chk(L.mastg_copy(ctx.h, dx, x.ctypes.data, x.nbytes, 0))
        ctx._chk(L.mastg_assemble(ctx.h, C.cast(dx, D), None, C.cast(dp.value + 16, D), mastg.DEVICE, 0))
        got = np.zeros_like(host)
        ctx._chk(L.mastg_copy(ctx.h, got.ctypes.data, dp, host.nbytes, 1))
    finally:
        L.mastg_device_free(ctx.h, dp)
        L.mastg_device_free(ctx.h, dx)
    assert np.array_equal(got[16:-16], J.view(np.uint8))
    assert (got[:16] == 0x5A).all() and (got[-16:] == 0x5A).all()
    ctx.close()
