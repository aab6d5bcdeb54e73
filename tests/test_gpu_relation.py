"""The tet-sphere relation at the edges of its kernel: neighbour lists
around the plane table's and the box polytope's capacities, one site, no
site near, ties, grids of one bin, and coordinates far from the origin or
of another scale.  The relation sets are compared with the oracle's."""
import dataclasses
import os
import sys

import numpy as np
import pytest
from scipy.spatial import cKDTree

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle  # noqa: E402
from libmat_amd import prep  # noqa: E402
from libmat_amd.rpd import Context  # noqa: E402
from rpd_compare import compare_relation, compare_with_oracle  # noqa: E402
from test_zz_no_alloc import _buffers, _out  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with Context(0) as c:
        yield c


def star(n):
    """One sphere in the middle with n neighbours around it."""
    k = np.arange(n) + 0.5
    ph, th = np.arccos(1 - 2 * k / n), np.pi * (1 + 5 ** 0.5) * k
    d = np.c_[np.cos(th) * np.sin(ph), np.sin(th) * np.sin(ph), np.cos(ph)]
    return np.c_[np.r_[[[0.5] * 3], 0.5 + 0.3 * d], np.full(n + 1, 0.01)]


def lattice(k):
    g = (np.arange(k) + 0.5) / k
    p = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    return np.c_[p, np.full(len(p), 0.05)]


def check(ctx, inst):
    orc = oracle.run(inst, mode=0)
    ctx.upload(inst)
    ctx.run()
    off, ids = ctx.relation()
    compare_relation(off, ids, orc)
    # (combinatorics: the relation decides which cells are clipped at all)
    compare_with_oracle(ctx.download(), orc, check_geometry=False)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 121, 122, 123, 127, 128,
                               129, 140])
def test_list_lengths(ctx, n):
    verts, tets = prep.grid_mesh(4, 0.1, n)
    check(ctx, prep.build_instance(verts, tets, star(n)))


@pytest.mark.parametrize("n,m", [(1, 1), (1, 40), (2, 1), (7, 3), (17, 1),
                                 (5, 900)])
def test_uneven_sizes(ctx, n, m):
    # one bin, one site, fewer tets than a wavefront, many sites per bin
    verts, tets = prep.grid_mesh(n, 0.1, n)
    check(ctx, prep.build_instance(verts, tets, prep.spheres(m, 0, n + m)))


@pytest.mark.parametrize("k", [2, 4])
def test_ties(ctx, k):
    # bisectors on the grid's planes and through its vertices
    verts, tets = prep.grid_mesh(4, 0.0, 0)
    check(ctx, prep.build_instance(verts, tets, lattice(k)))


@pytest.mark.parametrize("shift,scale", [(1000.0, 1.0), (-3.0e5, 1.0),
                                         (0.0, 1e-7), (2.0, 1e6)])
def test_frames(ctx, shift, scale):
    verts, tets = prep.grid_mesh(6, 0.1, 2)
    sph = prep.spheres(150, 0, 8)
    verts = verts * scale + shift
    sph = np.c_[sph[:, :3] * scale + shift, sph[:, 3] * scale]
    lo, hi = -1e-6 * scale + shift, (1 + 1e-6) * scale + shift
    check(ctx, prep.build_instance(verts, tets, sph,
                                   box=np.array([lo] * 3 + [hi] * 3)))


def far_frame(scale):
    """A small instance at a scale where the squares of its coordinates and
    the bisectors' constant terms approach or leave binary32's range."""
    verts, tets = prep.grid_mesh(6, 0.1, 2)
    inst = prep.build_instance(verts, tets, prep.spheres(150, 0, 8))
    return dataclasses.replace(
        inst, verts=inst.verts * scale,
        sites=inst.sites * np.array([scale] * 3 + [scale * scale]))


@pytest.mark.parametrize("scale", [1e17, 1e19, 5e19, 1e20, 1e25])
def test_frames_beyond_binary32(ctx, scale):
    check(ctx, far_frame(scale))


@pytest.mark.parametrize("scale", [1e17, 1e19, 5e19, 1e20, 1e25])
def test_proposal_frames_beyond_binary32(ctx, scale):
    # every proposal the plain relation holds passes the proposals' own test
    ctx.upload(far_frame(1.0))
    ctx.run(learned=2, proposal_k=32)
    want = ctx.stats()["learned"]
    proposed(ctx, far_frame(scale))
    assert ctx.stats()["learned"] == want


def proposed(ctx, inst):
    # proposals are tested with binary32 planes of their own: what they let
    # through is in the plain relation, and the cells are the plain path's
    ctx.upload(inst)
    ctx.run()
    off, ids = ctx.relation()
    want = ctx.download()
    pairs = set(zip(np.repeat(np.arange(inst.n_tet), np.diff(off)), ids))
    ctx.run(learned=2, proposal_k=32)
    off, ids = ctx.relation()
    assert set(zip(np.repeat(np.arange(inst.n_tet), np.diff(off)),
                   ids)) <= pairs
    got = ctx.download()
    for k in ("cells", "words", "geom", "areas"):
        assert np.array_equal(getattr(got, k), getattr(want, k))


@pytest.mark.parametrize("n", [1, 2, 63, 127, 128, 129, 140])
def test_proposal_list_lengths(ctx, n):
    verts, tets = prep.grid_mesh(4, 0.1, n)
    proposed(ctx, prep.build_instance(verts, tets, star(n)))


@pytest.mark.parametrize("shift,scale", [(0.0, 0.0), (1000.0, 1.0),
                                         (-3.0e5, 1.0), (0.0, 1e-7),
                                         (2.0, 1e6)])
def test_proposal_frames_and_ties(ctx, shift, scale):
    if scale == 0:  # ties: bisectors through the grid's vertices
        verts, tets = prep.grid_mesh(4, 0.0, 0)
        return proposed(ctx, prep.build_instance(verts, tets, lattice(4)))
    verts, tets = prep.grid_mesh(6, 0.1, 2)
    sph = prep.spheres(150, 0, 8)
    sph = np.c_[sph[:, :3] * scale + shift, sph[:, 3] * scale]
    lo, hi = -1e-6 * scale + shift, (1 + 1e-6) * scale + shift
    proposed(ctx, prep.build_instance(verts * scale + shift, tets, sph,
                                      box=np.array([lo] * 3 + [hi] * 3)))


def test_subsets_and_meshes_in_turn(ctx):
    # the tet order of the grid follows the mesh and the subset in use
    rng = np.random.default_rng(3)
    for n, m in ((6, 80), (9, 200), (6, 50)):
        verts, tets = prep.grid_mesh(n, 0.1, n + m)
        inst = prep.build_instance(verts, tets, prep.spheres(m, 0, m))
        ctx.upload(inst)
        ctx.run()
        off, ids = ctx.relation()
        for share in (0.5, 0.02, 1.0):
            sel = np.sort(rng.choice(inst.n_tet,
                                     max(1, int(share * inst.n_tet)),
                                     replace=False))
            ctx.set_tet_subset(sel)
            ctx.run()
            o2, i2 = ctx.relation()
            cnt = np.zeros(inst.n_tet, np.int64)
            cnt[sel] = np.diff(off)[sel]
            assert np.array_equal(np.diff(o2), cnt)
            assert np.array_equal(i2, np.concatenate(
                [ids[off[t]:off[t + 1]] for t in sel]))
        ctx.set_tet_subset(None)
        ctx.run()
        o2, i2 = ctx.relation()
        assert np.array_equal(off, o2) and np.array_equal(ids, i2)


def test_graph_follows_a_new_mesh_of_the_same_sizes(ctx):
    insts = []
    for seed, scale in ((1, 1.0), (2, 3.0)):
        verts, tets = prep.grid_mesh(6, 0.1, seed)
        sph = prep.spheres(40, 0, 5) * scale
        box = np.array([-1e-6 * scale] * 3 + [(1 + 1e-6) * scale] * 3)
        insts.append(prep.build_instance(verts * scale, tets, sph, box=box))
    assert insts[0].n_site == insts[1].n_site
    ctx.upload(insts[0])
    ctx.graph_build(headroom=1.0)
    for inst in (insts[1], insts[0], insts[0]):
        ctx.upload(inst)
        ctx.graph_run()
        got = ctx.download()
        ctx.run()
        want = ctx.download()
        assert np.array_equal(got.cells, want.cells)
        assert np.array_equal(got.words, want.words)
        assert np.array_equal(got.geom, want.geom)


@pytest.mark.parametrize("learned", [0, 2])
def test_graph_replays_on_meshes_of_the_same_sizes(ctx, learned):
    # and after an allocation-free call, which has an instance of its own
    small = prep.build_instance(*prep.grid_mesh(2, 0.1, 1),
                                prep.spheres(30, 0, 1))
    small.verts[:] *= 0.5
    insts = []
    for seed, scale in ((1, 1.0), (2, 1.0), (3, 4.0)):
        inst = prep.build_instance(*prep.grid_mesh(6, 0.1, seed),
                                   prep.spheres(40, 0, 5))
        insts.append(dataclasses.replace(
            inst, verts=inst.verts * scale,
            sites=inst.sites * np.array([scale] * 3 + [scale * scale])))
    ctx.upload(insts[0])
    ctx.graph_build(headroom=1.0, learned=learned)
    n = (1 << 13, 1 << 19, 1 << 17)
    bufs = _buffers(*n)
    for inst in insts[::-1] + insts:
        ctx.upload(inst)
        for _ in range(2):
            rc, _, err = ctx.run_noalloc(small, _out(bufs, *n))
            assert rc == 0, err
            _, replayed = ctx.graph_run()
            assert replayed
            got = ctx.download()
            ctx.run(learned=learned)
            want = ctx.download()
            for k in ("cells", "words", "geom", "areas"):
                assert np.array_equal(getattr(got, k), getattr(want, k))


@pytest.mark.parametrize("learned", [0, 2])
def test_graph_after_a_run_on_other_site_counts(ctx, learned):
    # the counts are the capture's again, the instance table in between was
    # not
    verts, tets = prep.grid_mesh(6, 0.1, 1)
    some = [[prep.sites_both(prep.spheres(m, 0, m))[1] for m in ms]
            for ms in ((40, 70), (300, 9))]
    adj = prep.tet_adjacency(verts.shape[0], tets)
    ctx.upload_batch([prep.Instance(verts, tets, *adj, *s) for s in some[0]])
    ctx.graph_build(headroom=1.0, learned=learned)
    for _ in range(2):
        ctx.update_sites_batch(some[1])
        ctx.run(learned=learned)
        ctx.update_sites_batch(some[0])
        ctx.graph_run()
        got = ctx.download()
        ctx.run(learned=learned)
        want = ctx.download()
        for k in ("cells", "words", "geom", "areas"):
            assert np.array_equal(getattr(got, k), getattr(want, k))


def unlisted(inst):
    """The same instance without neighbour lists: every sphere relates to
    every tet, far more pairs than a run expects of its sizes."""
    return dataclasses.replace(
        inst, knn_off=np.zeros(inst.n_site + 1, np.int64),
        knn_ids=np.zeros(0, np.int32))


def test_more_pairs_than_the_list_holds():
    verts, tets = prep.grid_mesh(6, 0.1, 2)
    inst = unlisted(prep.build_instance(verts, tets, prep.spheres(300, 0, 8)))
    with Context(0) as ctx:  # (a list of its own, as a first run finds it)
        ctx.upload(inst)
        st = [ctx.run(count_work=True) for _ in range(2)]
        off, ids = ctx.relation()
    n = inst.n_tet * inst.n_site
    for s in st:  # the first pass, which ran out of room, counts nothing
        assert s["n_candidates"] == n and s["relation_work"][0] == n
    assert st[0]["relation_work"] == st[1]["relation_work"]
    assert np.array_equal(off, np.arange(inst.n_tet + 1) * inst.n_site)
    assert np.array_equal(ids.reshape(inst.n_tet, -1),
                          np.tile(np.arange(inst.n_site), (inst.n_tet, 1)))


def test_more_pairs_than_a_captured_list_holds():
    verts, tets = prep.grid_mesh(6, 0.1, 2)
    few = prep.build_instance(verts, tets, prep.spheres(300, 0, 8))
    with Context(0) as ctx:
        for inst in (few, unlisted(few), few):
            ctx.upload(few)
            ctx.graph_build()
            ctx.update_sites(inst.sites, inst.flags, inst.knn_off,
                             inst.knn_ids)
            st, replayed = ctx.graph_run()
            assert replayed == (inst is few)
            got = ctx.download()
            ctx.run()
            want = ctx.download()
            for k in ("cells", "words", "geom", "areas"):
                assert np.array_equal(getattr(got, k), getattr(want, k))


def test_boxes_of_more_than_2_31_bins(ctx):
    # lists too long for the box polytope: every sphere's box is the domain,
    # 8,400 times 262,144 bins in all; the cells fill the cube
    verts, tets = prep.grid_mesh(64, 0.1, 3)
    n, k = 8400, 123
    p = np.random.default_rng(4).random((n, 3))
    ids = np.sort(cKDTree(p).query(p, k + 1)[1][:, 1:], axis=1)
    adj = prep.tet_adjacency(verts.shape[0], tets)
    ctx.upload(prep.Instance(verts, tets, *adj, np.c_[p, np.zeros(n)],
                             np.ones(n, np.uint32),
                             np.arange(n + 1, dtype=np.int64) * k,
                             ids.astype(np.int32).ravel()))
    st = ctx.run()
    assert st["n_bbox_fallback"] == n
    assert st["n_bin_registrations"] > 1 << 31
    assert abs(ctx.download().geom[:, 0].sum() - 1) < 1e-9


def graded(n, p, sph):
    """The grid with its corners' coordinates to the p-th power: most tets
    in few bins of the candidate grid."""
    verts, tets = prep.grid_mesh(n, 0.1, 3)
    return prep.build_instance(np.clip(verts, 0, 1) ** p, tets, sph)


@pytest.mark.parametrize("m", [1, 3, 40])
def test_graded_mesh(ctx, m):
    # rows of several thousand tets and rows of none: parts cut by count
    check(ctx, graded(20, 4, prep.spheres(m, 0, 5)))


def squeezed(n, p, scale, m):
    """The grid graded by the p-th power, then scaled per axis, and its
    spheres."""
    verts, tets = prep.grid_mesh(n, 0.1, 3)
    scale = np.asarray(scale, float)
    sph = prep.spheres(m, 0, 5)
    sph[:, :3] *= scale
    sph[:, 3] *= scale.min()
    return prep.build_instance(
        np.clip(verts, 0, 1) ** p * scale, tets, sph,
        box=np.r_[-1e-6 * scale, (1 + 1e-6) * scale])


@pytest.mark.parametrize("p", [1, 3])
@pytest.mark.parametrize("scale", [
    (0.02, 1, 1), (1, 0.02, 1), (1, 1, 0.02), (0.5, 0.02, 1), (1, 0.02, 0.02),
    (0.02, 1, 0.02), (0.02, 0.02, 1), (0.02, 0.5, 1)])
def test_flat_and_long_meshes(ctx, scale, p):
    # the grid's rows run along its longest axis
    check(ctx, squeezed(9, p, scale, 25))


@pytest.mark.parametrize("p", [1, 3])
@pytest.mark.parametrize("scale", [(0.002, 1, 1), (1, 0.002, 1)])
def test_relation_of_a_flat_mesh_is_spread_over_the_chip(ctx, scale, p):
    # (boxes and relation of one sphere took 7 to 15 ms, the clip 0.5)
    ctx.upload(squeezed(64, p, scale, 1))
    ms = np.array([ctx.run()["ms_kernel"] for _ in range(6)])
    assert (ms[:, 0] + ms[:, 2]).min() < ms[:, 5].min()


@pytest.mark.parametrize("p,m", [(1, 1), (1, 5), (4, 100)])
def test_relation_is_spread_over_the_chip(ctx, p, m):
    # few spheres, or most tets in few bins: the relation is no serial walk
    # of some wavefronts (3.7, 1.3 and 5.4 ms when it was; the clip takes
    # 0.4 to 0.7 ms, the relation a third of that)
    ctx.upload(graded(64, p, prep.spheres(m, 0, 5)))
    ms = np.array([ctx.run()["ms_kernel"] for _ in range(6)])
    assert ms[:, 2].min() < ms[:, 5].min()
