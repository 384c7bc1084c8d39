"""Jacobian values into the caller's device memory: the row assembly writes them
beside its own matrix, other assemblies and addresses that its kernels may not
write (not 8-byte aligned) take a copy.  Bitwise the host call's values,
whatever lies around them untouched, and the context's own matrix is the same."""
import ctypes as C

import numpy as np
import pytest

from helpers import ctx_from_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,mesh", [("hex8", (1, 1, 1)), ("hex8", (7, 5, 3)), ("distorted", (5, 4, 3)),
                                       ("plate", (6, 5)), ("heat", (4,))])
@pytest.mark.parametrize("shift", [0, 8, 4])      # bytes past an aligned address
def test_device_jacobian(oracle, mastg, kind, mesh, shift):
    print(f"[device J] {kind} {mesh} +{shift}", flush=True)
    if kind in ("hex8", "distorted"):
        P = oracle.Problem(oracle.CANTILEVER, *mesh, seed=5, lo=0.2, hi=1.0)
    elif kind == "plate":
        P = oracle.Problem(oracle.PLATE, *mesh, seed=5)
    else:
        P = oracle.Problem(oracle.HEAT, *mesh, seed=5)
    if kind == "distorted":
        xyz, conn = P.mesh()
        base, con = P.dofmap()
        xyz = xyz + np.random.default_rng(1).uniform(-0.01, 0.01, xyz.shape)
        desc = mastg.desc_from_arrays(mastg.HEX8_ELASTIC, xyz, conn, P.n_vars, node_dof_base=base,
                                      constrained_dofs=np.nonzero(con)[0], point_loads=P.point_load(), E=72e9,
                                      nu=0.33, penalty=3.0)
        ctx = mastg.Context(desc)
        ctx._keep = desc
        ctx.set_params(P.params())
    else:
        ctx = ctx_from_oracle(mastg, P)
    _, J = ctx.assemble()
    n = J.nbytes
    host = np.full(n + 64, 0x5A, np.uint8)
    L, dp = mastg.lib(), C.c_void_p()
    ctx._chk(L.mastg_device_alloc(ctx.h, host.nbytes, C.byref(dp)))
    try:
        ctx._chk(L.mastg_copy(ctx.h, dp, host.ctypes.data, host.nbytes, 0))
        ctx._chk(L.mastg_assemble(ctx.h, None, None, C.cast(dp.value + 16 + shift, C.POINTER(C.c_double)),
                                mastg.DEVICE, 0))
        got = np.zeros_like(host)
        ctx._chk(L.mastg_copy(ctx.h, got.ctypes.data, dp, host.nbytes, 1))
    finally:
        L.mastg_device_free(ctx.h, dp)
    a = 16 + shift
    assert np.array_equal(got[a:a + n].view(np.uint8), J.view(np.uint8))
    assert (got[:a] == 0x5A).all() and (got[a + n:] == 0x5A).all()
    x = np.random.default_rng(2).standard_normal(P.n_dofs)
    y = ctx.jacobian_product(x)
    ctx.assemble()
    assert np.array_equal(y, ctx.jacobian_product(x))
    ctx.close()
