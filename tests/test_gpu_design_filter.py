"""The filter by row patterns (meshes large enough for it, rows that lie together)
and by its CSR on either side of the rule between them, rows that are nearly
alike, and values that are no ordinary numbers, against numpy: a sum over the
neighbours' offsets on the box of elements."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _box(planes):
    """A box mesh with node planes at the given coordinates, x fastest."""
    nx, ny, nz = (len(p) - 1 for p in planes)
    z, y, x = np.meshgrid(planes[2], planes[1], planes[0], indexing="ij")
    xyz = np.stack([x, y, z], -1).reshape(-1, 3)
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    corner = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
    conn = np.stack([(i + a + (nx + 1) * (j + b + (ny + 1) * (k + c))).ravel() for a, b, c in corner], -1)
    return xyz, conn.astype(np.int32)


class _Filter:
    """W and its transpose on the box, neighbour by neighbour."""

    def __init__(self, planes, r):
        self.c = [(p[:-1] + p[1:]) / 2 for p in planes]
        self.shape = tuple(len(q) for q in self.c)
        self.r = r
        m = [min(int(np.ceil(r / np.diff(p).min())), len(q) - 1) for p, q in zip(planes, self.c)]
        self.off = list(itertools.product(*[range(-a, a + 1) for a in m]))
        self.S = self._sum(np.ones(self.shape))

    def _sum(self, x):
        y = np.zeros(self.shape)
        for o in self.off:
            dst = tuple(slice(max(0, -a), n - max(0, a)) for a, n in zip(o, self.shape))
            src = tuple(slice(max(0, a), n - max(0, -a)) for a, n in zip(o, self.shape))
            d2 = 0.0
            for k in range(3):
                d = self.c[k][src[k]] - self.c[k][dst[k]]
                d2 = d2 + (d * d).reshape([-1 if q == k else 1 for q in range(3)])
            w = self.r - np.sqrt(d2)
            with np.errstate(invalid="ignore"):
                y[dst] += np.where(w >= 0, w * x[src], 0.0)
        return y

    def __call__(self, x, transpose):
        x = x.reshape(self.shape[::-1]).transpose(2, 1, 0)
        y = self._sum(x / self.S) if transpose else self._sum(x) / self.S
        return y.transpose(2, 1, 0).ravel()


def _design(mastg, planes, r):
    xyz, conn = _box(planes)
    return mastg.Design(mastg.desc_from_arrays(mastg.HEX8_ELASTIC, xyz, conn, 6), r)


def _planes(mesh, graded=""):
    rng = np.random.default_rng(6)
    return [np.arange(n + 1.0) + (rng.integers(-8, 9, n + 1) / 256.0 if a in graded else 0.0) for n, a in zip(mesh, "xyz")]


# by patterns: rows of 7, 27, 33 and 81 neighbours, last waves with few rows
# (odd counts), rows of elements that are no whole lines, many short groups
# (graded along z); by the CSR: too small, graded along x (rows of a pattern far
# apart), too many patterns (along y and z)
@pytest.mark.parametrize("mesh,r,graded", [((128, 41, 35), 1.05, ""), ((65, 33, 25), 1.8, ""), ((40, 51, 63), 2.05, ""),
                                           ((41, 37, 43), 2.55, ""), ((51, 43, 41), 2.55, "z"),
                                           ((23, 21, 19), 2.55, ""), ((64, 33, 31), 2.55, "x"),
                                           ((40, 41, 43), 1.55, "yz")])
def test_filter_on_either_side_of_the_rule(mastg, mesh, r, graded):
    """Bar 2e-13, 0.1 of: weights shared to 16 eps of the largest coordinate, 128 at most
    (4.6e-13), over the mean weight of a row (r / 4 at least, 0.5 of a cell), and
    the inputs' spread about their mean; the sums themselves to 100 eps."""
    print(f"[filter rule] {mesh} r = {r} graded {graded!r}", flush=True)
    planes = _planes(mesh, graded)
    Dg, F = _design(mastg, planes, r), _Filter(planes, r)
    x = np.random.default_rng(1).uniform(0.9, 1.1, np.prod(mesh))
    for t in (False, True):
        y = F(x, t)
        assert np.max(np.abs(Dg.filter(x, transpose=t) - y)) <= 2e-13 * np.abs(y).max()
    Dg.close()


@pytest.mark.parametrize("origin", [0.0, 2.0 ** 20])
def test_rows_that_nearly_agree(mastg, origin):
    """Planes of nodes displaced by -2^-29, 0 or 2^-29 (1.9e-9 of a cell) along z:
    at 2^20 from the origin that is eight units of the coordinates' rounding, sums
    of eight of them are exact, and so are the centroids: a row's weights are
    known to 1e-15, and the filter's values to 1e-12 (weights may be shared to
    2^-40 of the radius: 0.9e-12 of it, times at most 4 for the ratio of the
    radius to the mean weight, times the inputs' spread of 0.1)."""
    print(f"[filter, rows nearly alike] origin {origin}", flush=True)
    mesh = (64, 35, 41)
    planes = [np.arange(n + 1.0) + origin for n in mesh]
    planes[2] += np.random.default_rng(8).integers(-1, 2, mesh[2] + 1) * 2.0 ** -29
    r = 2.2
    Dg, F = _design(mastg, planes, r), _Filter(planes, r)
    x = np.random.default_rng(1).uniform(0.9, 1.1, np.prod(mesh))
    for t in (False, True):
        y = F(x, t)
        assert np.max(np.abs(Dg.filter(x, transpose=t) - y)) <= 1e-12 * np.abs(y).max()
    Dg.close()


# patterns of 7 (padded by 9 to a batch of 16), 27 and 33 neighbours; the CSR
@pytest.mark.parametrize("mesh,r", [((128, 41, 35), 1.05), ((65, 33, 25), 1.8), ((64, 35, 41), 2.05), ((9, 8, 7), 1.8)])
def test_infinities_stay_where_they_belong(mastg, mesh, r):
    """An infinite input makes the rows that hold it infinite, of its sign, and no
    others; NaN likewise: as a sum over the row's neighbours gives it."""
    print(f"[filter, infinities] {mesh} r = {r}", flush=True)
    planes = _planes(mesh)
    Dg, F = _design(mastg, planes, r), _Filter(planes, r)
    rng = np.random.default_rng(3)
    n = int(np.prod(mesh))
    for bad in (np.inf, -np.inf, np.nan):
        x = rng.uniform(0.1, 1.0, n)
        x[[0, n // 2, n - 1]] = bad
        for t in (False, True):
            y, z = F(x, t), Dg.filter(x, transpose=t)
            assert np.array_equal(np.isnan(z), np.isnan(y)) and np.array_equal(np.isinf(z), np.isinf(y))
            assert np.array_equal(z[np.isinf(y)], y[np.isinf(y)])
            ok = np.isfinite(y)
            assert np.max(np.abs(z[ok] - y[ok])) <= 1e-12 * np.abs(y[ok]).max()
    Dg.close()
