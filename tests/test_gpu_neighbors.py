"""The device neighbour builder at the edges of its tiers: sets smaller than
a candidate batch, cells that outgrow the small tier's 64 vertices, cells
over the builder's capacities, and ties (bisectors through one point)."""
import numpy as np
import pytest

from libmat_amd import prep
from libmat_amd.rpd import Context

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with Context(0) as c:
        yield c


def star(n):
    """One sphere at the centre and n around it on a sphere: its cell has n
    facets and 2 n - 4 vertices."""
    k = np.arange(n) + 0.5
    ph, th = np.arccos(1 - 2 * k / n), np.pi * (1 + 5 ** 0.5) * k
    d = np.c_[np.cos(th) * np.sin(ph), np.sin(th) * np.sin(ph), np.cos(ph)]
    xyz = np.r_[[[0.5, 0.5, 0.5]], 0.5 + 0.3 * d]
    return np.c_[xyz, np.full(n + 1, 1e-4)]


@pytest.mark.parametrize("n", [1, 2, 3, 63, 65, 129])
def test_small_sets(ctx, n):
    xyzw = prep.spheres(n, 0, 40 + n)
    xyzw[:, 3] **= 2
    want = prep.power_neighbors(xyzw, prep.UNIT_BOX)
    got = ctx.power_neighbors(xyzw, prep.UNIT_BOX)
    for a, b in zip(want, got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [33, 34, 80, 129])
def test_cells_over_the_small_tier(ctx, n):
    xyzw = star(n)
    want = prep.power_neighbors(xyzw, prep.UNIT_BOX)
    got = ctx.power_neighbors(xyzw, prep.UNIT_BOX)
    assert want[1][1] == n  # the centre names every other sphere
    for a, b in zip(want, got):
        assert np.array_equal(a, b)


def test_cells_over_the_capacities_are_refused(ctx):
    with pytest.raises(RuntimeError, match="exceeds the cell capacities"):
        ctx.power_neighbors(star(200), prep.UNIT_BOX)
    # and the context goes on
    xyzw = star(20)
    assert np.array_equal(ctx.power_neighbors(xyzw, prep.UNIT_BOX)[2],
                          prep.power_neighbors(xyzw, prep.UNIT_BOX)[2])


@pytest.mark.parametrize("k", [3, 5])
def test_lattice_ties(ctx, k):
    # equal spheres on a lattice: every vertex of a cell lies on bisectors
    # of spheres that touch the cell there only; which of them are listed
    # follows from the order of the search, but the face neighbours always
    # are, nothing past the next shell is, and the lists are symmetric
    g = (np.arange(k) + 0.5) / k
    p = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    xyzw = np.c_[p, np.full(len(p), 1e-3)]
    valid, off, ids, _ = ctx.power_neighbors(xyzw, prep.UNIT_BOX)
    assert (valid == 1).all()
    d = np.abs(p[:, None] - p[None]).round(9)
    face = np.isclose(d.sum(-1), 1 / k)
    near = d.max(-1) < 1.01 / k
    for i in range(len(p)):
        mine = ids[off[i]:off[i + 1]]
        assert (np.diff(mine) > 0).all() and near[i][mine].all()
        assert set(np.nonzero(face[i])[0]) <= set(mine)
        assert all(i in ids[off[j]:off[j + 1]] for j in mine)


@pytest.mark.parametrize("shift", [0.0, 1000.0])
@pytest.mark.parametrize("kind", ["slab", "line", "corners"])
def test_cells_that_reach_far_on_one_side(ctx, kind, shift):
    # shells of many grid cells of which a one-sided or flat cell needs a
    # few rows: spheres near a face of the box, along a diagonal, and in two
    # small clusters of different weight classes (each outside the other's
    # grid); general position, so the lists are the host builder's
    rng = np.random.default_rng(11)
    p = rng.random((400, 3))
    w = np.full(400, 1e-4) * (1 + rng.random(400))
    if kind == "slab":
        p[:, 2] = 0.02 + 0.001 * p[:, 2]
    elif kind == "line":
        p = 0.1 + 0.8 * p[:, :1] + 0.002 * p
    else:
        p = np.where(np.arange(400)[:, None] < 200, 0.05 + 0.02 * p,
                     0.9 + 0.03 * p)
        w[:200] *= 1e-2
    box = np.asarray(prep.UNIT_BOX) + shift
    xyzw = np.c_[p + shift, w]
    want = prep.power_neighbors(xyzw, box)
    got = ctx.power_neighbors(xyzw, box)
    for a, b in zip(want, got):
        assert np.array_equal(a, b)


def test_scale_and_offset_are_free(ctx):
    # powers of two keep every bit, so the lists are the same; neither they
    # nor an offset leave more signs to the exact predicates (6,000 spheres
    # took 10 ms at unit scale and 50 to 2,500 ms in these frames)
    xyzw = prep.spheres(6000, 1, 7)
    xyzw[:, 3] **= 2
    box = np.asarray(prep.UNIT_BOX)
    want = ctx.power_neighbors(xyzw, box)

    def ms(x, b):
        return min(ctx.power_neighbors(x, b)[3] for _ in range(3))

    limit = 2.5 * ms(xyzw, box)
    for e in (-33, 50, 60, 66, 73):
        s = 2.0 ** e
        x = xyzw * np.array([s, s, s, s * s])
        got = ctx.power_neighbors(x, box * s)
        for a, b in zip(want[:3], got[:3]):
            assert np.array_equal(a, b)
        assert ms(x, box * s) < limit, e
    x = xyzw + np.array([1e6, 1e6, 1e6, 0])
    assert ms(x, box + 1e6) < limit
