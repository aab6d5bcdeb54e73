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
