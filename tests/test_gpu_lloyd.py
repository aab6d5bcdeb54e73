"""The Lloyd step's kernels where they branch: sites around and over one
wavefront's share of cells, and site sets that keep hidden spheres."""
import numpy as np
import pytest

from libmat_amd import prep
from libmat_amd.rpd import Context

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with Context(0) as c:
        yield c


@pytest.mark.parametrize("n,m", [(8, 1), (9, 1), (9, 2), (16, 1), (20, 3),
                                 (24, 40)])
def test_centroids_of_large_sites(ctx, n, m):
    # 3,072 to 82,944 cells, all in one site or spread over a few: 64-bit
    # sums of at most 10^5 positive terms, so 1e-11 of the value
    verts, tets = prep.grid_mesh(n, 0.1, n)
    inst = prep.build_instance(verts, tets, prep.spheres(m, 0, n + m))
    ctx.upload(inst)
    ctx.run()
    res = ctx.download()
    got = ctx.site_centroids()
    want = np.c_[inst.sites[:, :3], np.zeros(inst.n_site)]
    for s in range(inst.n_site):
        g = res.geom[res.cells["seed"] == s]
        if g.size and g[:, 0].sum() != 0:
            want[s, 3] = g[:, 0].sum()
            want[s, :3] = (g[:, :1] * g[:, 1:]).sum(0) / want[s, 3]
    assert np.allclose(got, want, rtol=1e-11, atol=1e-11)
    assert np.array_equal(got, ctx.site_centroids())


@pytest.mark.parametrize("rule,m", [(1, 400), (2, 900), (0, 3), (0, 1)])
def test_owners_with_hidden_spheres_kept(ctx, rule, m):
    # every sphere a site, hidden ones unflagged with an empty list: a tet's
    # proposals hold the visible sphere that owns its centroid
    verts, tets = prep.grid_mesh(7, 0.1, 3)
    xyzr = prep.spheres(m, rule, 60 + m)
    compact, every = prep.sites_both(xyzr)
    inst = prep.build_instance(verts, tets, xyzr)
    inst.sites, inst.flags, inst.knn_off, inst.knn_ids = every
    ctx.upload(inst)
    knn, _ = ctx.features()
    c = verts[tets].mean(1)
    s, vis = every[0], np.nonzero(every[1])[0]
    pd = ((c[:, None] - s[None, vis, :3]) ** 2).sum(-1) - s[None, vis, 3]
    # (the five owners of a tet tie for the first slots)
    assert (knn == vis[pd.argmin(1)][:, None]).any(1).all()
    assert (every[1][knn[:, 0]] == 1).all()
    # and the cells are the plain path's
    ctx.run(learned=2, proposal_k=8)
    a = ctx.download()
    ctx.run()
    b = ctx.download()
    assert np.array_equal(a.cells, b.cells) and np.array_equal(a.geom, b.geom)
