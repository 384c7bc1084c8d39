"""The optimality-criteria step where a wave of the candidate sweep takes several
batches of 64 elements (more than 131,072 elements: a full batch and one, a full
batch and a few, exactly one batch) and where a few work-groups' partial sums
meet with ragged last shares, against the oracle's bisection.  Bars as for the
small meshes: densities 1e-8 (the multiplier comes from a 7-pass multi-section
to ~1e-10 relative), volume 1e-8 of the total."""
import numpy as np
import pytest

import design as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", [(129, 33, 31), (83, 41, 41), (64, 64, 32), (17, 11, 13), (27, 19, 19)])
def test_oc_update_batches(oracle, mastg, mesh):
    print(f"[design OC] hex8 {mesh}", flush=True)
    P = oracle.Problem(oracle.CANTILEVER, *mesh, seed=2, lo=0.3, hi=1.0)
    xyz, conn = P.mesh()
    Dg = mastg.Design(mastg.desc_from_arrays(mastg.HEX8_ELASTIC, xyz, conn, P.n_vars), 0.6 / mesh[0])
    n = P.n_elems
    rng = np.random.default_rng(5)
    rho = rng.uniform(0.05, 0.95, n)
    # sensitivities that depend on the place: an element left out, taken twice
    # or weighted with a neighbour's values changes the volumes
    dc = -10.0 ** rng.uniform(-3, 2, n)
    Ve = D.hex8_volumes(xyz, conn) * (1.0 + np.arange(n) / n)
    vf, move, rmin = 0.4 * Ve.sum() / Dg.v_total, 0.2, 1e-3
    new, lam = Dg.oc_update(rho, dc, Ve, vf, move, rmin)
    ref, lam0 = D.oc_update(rho, dc, Ve, Dg.v_total, vf, move, rmin)
    err = np.max(np.abs(new - ref))
    print(f"  lambda {lam:.12e} (oracle {lam0:.12e}), max |rho - oracle| {err:.2e}", flush=True)
    assert err <= 1e-8
    assert abs(np.dot(Ve, new) - vf * Dg.v_total) <= 1e-8 * Ve.sum()
    Dg.close()
