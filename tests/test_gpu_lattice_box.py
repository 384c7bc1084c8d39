"""The hex8 lattice operator of axis-aligned boxes (modes of the class matrix)
and, on sheared cells, the general form it stands beside: the operator against
the assembled CSR (1e-12 of max |y|, the bar of every operator), and the
multigrid design evaluation against Jacobi-CG on the assembled matrix
(compliance 1e-9, gradient 1e-7)."""
import numpy as np
import pytest

from helpers import ctx_from_oracle, rel_err_floor

pytestmark = pytest.mark.gpu


# a wave owns 62 points of an x-y plane: planes of 63 (one point over), 123
# (one short of two waves), 125, 21 (a third of one) and 825 points; cells
# that are no cubes
@pytest.mark.parametrize("mesh", [(8, 6, 4), (40, 2, 2), (24, 4, 6), (6, 2, 2), (32, 24, 8)])
def test_box_operator_equals_csr(oracle, mastg, mesh):
    print(f"[box operator] {mesh}", flush=True)
    P = oracle.Problem(oracle.CANTILEVER, *mesh, seed=4, lo=0.01, hi=1.0)
    ctx = ctx_from_oracle(mastg, P)
    ctx.assemble()
    _, con = P.dofmap()
    x = np.random.default_rng(7).standard_normal(P.n_dofs)
    y0 = ctx.jacobian_product(np.where(con == 1, 0.0, x), op=0)
    y3 = ctx.jacobian_product(x, op=3)
    assert np.max(np.abs(y3 - y0)) <= 1e-12 * np.max(np.abs(y0))
    ctx.close()


def _sheared(mastg, oracle, mesh, shear):
    P = oracle.Problem(oracle.CANTILEVER, *mesh, seed=4, lo=0.1, hi=1.0)
    xyz, conn = P.mesh()
    base, con = P.dofmap()
    xyz = xyz.copy()
    xyz[:, 0] += shear * xyz[:, 2]
    desc = mastg.desc_from_arrays(mastg.HEX8_ELASTIC, xyz, conn, P.n_vars, node_dof_base=base,
                                  constrained_dofs=np.nonzero(con)[0], point_loads=P.point_load(), E=72e9, nu=0.33,
                                  penalty=3.0)
    ctx = mastg.Context(desc)
    ctx._keep = desc
    ctx.set_params(P.params())
    return P, con, ctx


@pytest.mark.parametrize("mesh,shear", [((8, 4, 4), 0.3), ((16, 8, 8), 0.5)])
def test_sheared_lattice(oracle, mastg, mesh, shear):
    print(f"[sheared lattice] {mesh} {shear}", flush=True)
    P, con, ctx = _sheared(mastg, oracle, mesh, shear)
    ctx.assemble()
    x = np.random.default_rng(7).standard_normal(P.n_dofs)
    y0 = ctx.jacobian_product(np.where(con == 1, 0.0, x), op=0)
    y3 = ctx.jacobian_product(x, op=3)
    assert np.max(np.abs(y3 - y0)) <= 1e-12 * np.max(np.abs(y0))
    ref = ctx.design_eval(P.params())
    r = ctx.design_eval(P.params(), solver=mastg.SOLVER_MG)
    assert r["rel_res"] <= 1.5e-10 and r["iters"] * 4 < ref["iters"], (r["iters"], ref["iters"])
    assert abs(r["objective"] - ref["objective"]) <= 1e-9 * abs(ref["objective"])
    assert rel_err_floor(r["grad"], ref["grad"], floor=1e-6) <= 1e-7
    ctx.close()


@pytest.mark.parametrize("steps", [1, 2, 8])
def test_box_smoothing_steps(oracle, mastg, steps):
    """The fewest, the shortest recurrence and the most smoothing passes; an odd
    number of iterations between polls and a replayed graph."""
    print(f"[box smoothing steps] {steps}", flush=True)
    P = oracle.Problem(oracle.CANTILEVER, 16, 8, 8, seed=3, lo=0.1, hi=1.0)
    ref = P.solve_elastic(1e-10)
    ctx = ctx_from_oracle(mastg, P)
    ctx.set_option(mastg.OPT_MG_STEPS_FINE, steps)
    for every in (0, 3):
        r = ctx.design_eval(P.params(), solver=mastg.SOLVER_MG, check_every=every)
        assert r["rel_res"] <= 1.5e-10
        assert abs(r["objective"] - ref["compliance"]) <= 1e-9 * abs(ref["compliance"])
        assert rel_err_floor(r["grad"], ref["dc"], floor=1e-6) <= 1e-7
    ctx.close()


# lattices that do not coarsen, down to one cell; rows of 62 and 63 points (a
# wave's share and one over); nodes and elements as the mesh generator numbers
# them and shuffled
@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("mesh", [(1, 1, 1), (3, 1, 1), (2, 3, 1), (7, 9, 11), (61, 2, 2), (62, 3, 1), (45, 23, 23)])
def test_matrix_free_cg_equals_csr_cg(oracle, mastg, mesh, shuffle):
    """Matrix-free CG on equal boxes runs the lattice product with its vectors
    in lattice order: the same Krylov iteration as on the assembled CSR, and
    the same answers."""
    print(f"[matrix-free CG] {mesh} shuffle={shuffle}", flush=True)
    P = oracle.Problem(oracle.CANTILEVER, *mesh, seed=4, lo=0.1, hi=1.0)
    xyz, conn = P.mesh()
    base, con = P.dofmap()
    rng = np.random.default_rng(11)
    if shuffle:
        node = rng.permutation(len(xyz))            # new node of each old one
        elem = rng.permutation(len(conn))
        xyz2, base2 = np.empty_like(xyz), np.empty_like(base)
        xyz2[node], base2[node] = xyz, base
        xyz, base, conn = xyz2, base2, node[conn][elem].astype(conn.dtype)
    desc = mastg.desc_from_arrays(mastg.HEX8_ELASTIC, xyz, conn, P.n_vars, node_dof_base=base,
                                  constrained_dofs=np.nonzero(con)[0], point_loads=P.point_load(), E=72e9, nu=0.33,
                                  penalty=3.0)
    ctx = mastg.Context(desc)
    ctx._keep = desc
    rho = rng.uniform(0.1, 1.0, len(conn))
    ref = ctx.design_eval(rho)
    for _ in range(2):                               # the first solve finds the lattice
        r = ctx.design_eval(rho, solver=mastg.SOLVER_MATFREE)
        assert r["rel_res"] <= 1.5e-10
        assert abs(r["iters"] - ref["iters"]) <= 2 + ref["iters"] // 50, (r["iters"], ref["iters"])
        assert abs(r["objective"] - ref["objective"]) <= 1e-9 * abs(ref["objective"])
        assert rel_err_floor(r["grad"], ref["grad"], floor=1e-6) <= 1e-7
    ctx.close()
