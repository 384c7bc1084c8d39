"""A Krylov solve that breaks down returns its error with the last iterate, the
same on every run and for every chunk of iterations between the host's looks: no
work-group goes on with the vectors once another has seen the breakdown.

The matrix is made indefinite by the material: at nu = 0.9 lambda + 2 G < 0, so
every field u_x(x) has negative energy (trilinear cells hold it exactly), while
the diagonal, (lambda + 2 G) + 2 G > 0 on cubes, and with it the Jacobi
preconditioner, stay positive: CG meets p.q <= 0 once its space holds such a
direction."""
import numpy as np
import pytest

from helpers import ctx_from_oracle

pytestmark = pytest.mark.gpu


# one work-group in the vector kernels, and more than the chip holds waves at
# once; a lattice (box product) and the assembled operator; PCG's update
@pytest.mark.parametrize("mesh,solver", [
    ((4, 2, 2), "SOLVER_CG_JACOBI"), ((48, 24, 24), "SOLVER_CG_JACOBI"), ((48, 24, 24), "SOLVER_MATFREE"),
    ((16, 8, 8), "SOLVER_MG"),
])
def test_breakdown_keeps_the_last_iterate(oracle, mastg, mesh, solver):
    print(f"[breakdown] {mesh} {solver}", flush=True)
    P = oracle.Problem(oracle.CANTILEVER, *mesh, seed=2, lo=0.3, hi=1.0)
    ctx = ctx_from_oracle(mastg, P, nu=0.9)
    R, _ = ctx.assemble()
    b = -R
    opts = dict(solver=getattr(mastg, solver), rtol=1e-12, raise_on_error=False)
    x, st = ctx.solve(b, check_every=1, **opts)
    assert st["rc"] == -4, st
    n = st["iters"]
    if solver != "SOLVER_MG":       # (its preconditioner may be indefinite from the start)
        assert n >= 1, st
    for every in (1, 4, 32):
        y, sy = ctx.solve(b, check_every=every, **opts)
        assert sy["rc"] == -4 and sy["iters"] == n and np.array_equal(x, y), (every, sy)
    if n:
        y, sy = ctx.solve(b, check_every=1, max_iters=n, **opts)
        assert sy["iters"] == n and np.array_equal(x, y), sy
    else:
        assert not x.any()
    ctx.close()
