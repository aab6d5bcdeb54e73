"""The training step at the edges of its tiles and chunks: batches of one
tile, of part of a weight-gradient chunk and of several, row counts that do
not fill the last batch.  The gradient is compared with the oracle's
(tolerances of the 16-bit layers: 2e-2 of a layer's largest gradient)."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import mlp_oracle  # noqa: E402
from libmat_amd import prep  # noqa: E402
from libmat_amd.rpd import Context  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with Context(0) as c:
        verts, tets = prep.grid_mesh(6, 0.1, 1)  # 1,296 rows
        c.upload(prep.build_instance(verts, tets, prep.spheres(90, 0, 2)))
        c.run()
        c.features(download=False)
        c.labels(download=False)
        yield c


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 127, 128, 129, 300])
def test_gradient_at_tile_edges(ctx, rows):
    _, X = ctx.features()
    Y, M = ctx.labels()
    ctx.mlp_init(rows)
    P = ctx.mlp_get()
    g, loss = ctx.mlp_grad(P, X[:rows], Y[:rows], M[:rows], 4.0)
    want_loss, want = mlp_oracle.loss_and_grad(
        P.astype(np.float64), mlp_oracle.from_bits(X[:rows]), Y[:rows],
        M[:rows], 4.0, True)
    assert abs(loss - want_loss) <= 1e-4 * max(1.0, abs(want_loss))
    a, b = mlp_oracle.unpack(g.astype(np.float64)), mlp_oracle.unpack(want)
    for name, _ in mlp_oracle.SHAPES:
        err = np.abs(a[name] - b[name]).max()
        assert err <= 2e-2 * np.abs(b[name]).max(), name


@pytest.mark.parametrize("batch", [16, 112, 128, 1024, 2048])
def test_training_is_repeatable_and_learns(ctx, batch):
    out = []
    for _ in range(2):
        ctx.mlp_init(3)
        loss = ctx.train(epochs=3, batch=batch, seed=9)
        out.append((loss, ctx.mlp_get()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
    assert np.isfinite(out[0][0]).all() and out[0][0][2] < out[0][0][0]
