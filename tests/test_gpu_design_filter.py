"""The filter's row patterns where rows are nearly alike or hold values that are
no ordinary numbers, against numpy on the same centroids."""
import numpy as np
import pytest

import design as D

pytestmark = pytest.mark.gpu


def _box(mesh):
    nx, ny, nz = mesh
    i, j, k = np.meshgrid(np.arange(nx + 1), np.arange(ny + 1), np.arange(nz + 1), indexing="ij")
    xyz = np.stack([i, j, k], -1).transpose(2, 1, 0, 3).reshape(-1, 3).astype(float)
    p = lambda a, b, c: a + (nx + 1) * (b + (ny + 1) * c)
    e = np.array([(a, b, c) for c in range(nz) for b in range(ny) for a in range(nx)])
    corner = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
    conn = np.stack([p(e[:, 0] + a, e[:, 1] + b, e[:, 2] + c) for a, b, c in corner], -1)
    return xyz, conn.astype(np.int32)


def _filter(mastg, xyz, conn, r):
    return mastg.Design(mastg.desc_from_arrays(mastg.HEX8_ELASTIC, xyz, conn, 6), r)


@pytest.mark.parametrize("origin", [0.0, 2.0 ** 20])
def test_rows_that_nearly_agree(mastg, origin):
    """Planes of nodes displaced by -2^-29, 0 or 2^-29 (1.9e-9 of a cell): at 2^20
    from the origin that is four units of the coordinates' rounding, sums of
    eight of them are exact, and so are the centroids: a row's weights are known
    to 1e-15, and the filter's values to 1e-12 (weights may be shared to 2^-40 of
    the radius: 0.9e-12 of it, times at most 3 for the ratio of the radius to the
    mean weight, times the inputs' spread of 0.2)."""
    print(f"[filter, rows nearly alike] origin {origin}", flush=True)
    mesh = (24, 6, 5)
    xyz, conn = _box(mesh)
    rng = np.random.default_rng(8)
    for d in range(3):
        step = rng.integers(-1, 2, mesh[d] + 1) * 2.0 ** -29
        xyz[:, d] += step[xyz[:, d].astype(int)]
    xyz += origin
    r = 2.2
    Dg = _filter(mastg, xyz, conn, r)
    W = D.filter_matrix(xyz[conn].sum(axis=1) / 8.0, r)
    x = rng.uniform(0.9, 1.1, len(conn))
    for t, M in ((False, W), (True, W.T)):
        y = M @ x
        assert np.max(np.abs(Dg.filter(x, transpose=t) - y)) <= 1e-12 * np.abs(y).max()
    Dg.close()


# rows of 1 (padded by 15 to a batch), 16 (none), 17 and up to 27 neighbours
@pytest.mark.parametrize("mesh,r", [((9, 1, 1), 0.5), ((16, 1, 1), 20.0), ((17, 1, 1), 20.0), ((9, 8, 7), 1.8)])
def test_infinities_stay_where_they_belong(mastg, mesh, r):
    """An infinite input makes the rows that hold it infinite, of its sign, and no
    others; NaN likewise: as a sum over the row's neighbours gives it."""
    print(f"[filter, infinities] {mesh} r = {r}", flush=True)
    xyz, conn = _box(mesh)
    Dg = _filter(mastg, xyz, conn, r)
    W = D.filter_matrix(D.centroids(xyz, conn), r)
    rng = np.random.default_rng(3)
    n = len(conn)
    for bad in (np.inf, -np.inf, np.nan):
        x = rng.uniform(0.1, 1.0, n)
        x[n // 2] = bad
        for t, M in ((False, W), (True, W.T)):
            y = np.array([sum(M[e, f] * x[f] for f in np.nonzero(M[e])[0]) for e in range(n)])
            z = Dg.filter(x, transpose=t)
            assert np.array_equal(np.isnan(z), np.isnan(y)) and np.array_equal(np.isinf(z), np.isinf(y))
            assert np.array_equal(z[np.isinf(y)], y[np.isinf(y)])
            ok = np.isfinite(y)
            assert not ok.any() or np.max(np.abs(z[ok] - y[ok])) <= 1e-13 * np.abs(y[ok]).max()
    Dg.close()
