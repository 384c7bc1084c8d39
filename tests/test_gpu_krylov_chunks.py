"""Krylov iterations run in chunks between the host's looks at the device
scalars, and each kernel sums the scalars of the one before it: where a chunk
ends must not show.  Any chunk length gives the same iterates (bitwise), the
same count, and an iteration limit stops every solver at exactly that count."""
import numpy as np
import pytest

from helpers import ctx_from_oracle

pytestmark = pytest.mark.gpu


def _system(oracle, mastg, kind):
    if kind == "hex8":
        P = oracle.Problem(oracle.CANTILEVER, 9, 5, 3, seed=2, lo=0.1, hi=1.0)
    elif kind == "hex8 lattice":
        P = oracle.Problem(oracle.CANTILEVER, 8, 4, 4, seed=2, lo=0.1, hi=1.0)
    elif kind == "plate":
        P = oracle.Problem(oracle.PLATE, 8, 8, seed=2)
    else:
        P = oracle.Problem(oracle.HEAT, 8, seed=2)
    ctx = ctx_from_oracle(mastg, P)
    R, _ = ctx.assemble()
    return ctx, -R


@pytest.mark.parametrize("kind,solver", [
    ("hex8", "SOLVER_CG_JACOBI"), ("hex8", "SOLVER_MATFREE"), ("hex8", "SOLVER_MIXED"),
    ("hex8 lattice", "SOLVER_MATFREE"), ("hex8 lattice", "SOLVER_MG"),
    ("plate", "SOLVER_CG_JACOBI"), ("plate", "SOLVER_MG"),
    ("heat", "SOLVER_BICGSTAB"),
])
def test_chunk_length_does_not_show(oracle, mastg, kind, solver):
    print(f"[krylov chunks] {kind} {solver}", flush=True)
    ctx, b = _system(oracle, mastg, kind)
    opts = dict(solver=getattr(mastg, solver), rtol=1e-8)
    x, st = ctx.solve(b, check_every=1, **opts)
    assert st["iters"] > 1 and st["rel_res"] <= 1.5e-8
    # the reduced-precision product replaces residuals at chunk ends: its
    # iterates may depend on the chunk, its answer may not
    for every in (2, 5, 32):
        y, sy = ctx.solve(b, check_every=every, **opts)
        if solver == "SOLVER_MIXED":
            assert sy["rel_res"] <= 1.5e-8
        else:
            assert sy["iters"] == st["iters"] and np.array_equal(x, y), (every, sy["iters"], st["iters"])
    n = max(1, st["iters"] - 1)
    xs = []
    for every in (1, 3, 32):
        y, sy = ctx.solve(b, max_iters=n, check_every=every, raise_on_error=False, **opts)
        assert sy["rc"] == -3 and sy["iters"] == n, (every, sy)
        xs.append(y)
    if solver != "SOLVER_MIXED":
        assert all(np.array_equal(xs[0], y) for y in xs[1:])
    z, sz = ctx.solve(np.zeros_like(b), **opts)
    assert sz["iters"] == 0 and not z.any()
    ctx.close()
