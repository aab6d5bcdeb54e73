"""The clip's cavity boundary in every shape: cells of few and of many planes
(the packed cycle in shapes of up to 16 planes, the serial walk above),
facets cut off altogether, and ties, against the oracle's serial walk."""
import os
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "oracle"))
import oracle  # noqa: E402
from libmat_amd import prep  # noqa: E402
from libmat_amd.rpd import Context  # noqa: E402
from rpd_compare import compare_with_oracle  # noqa: E402

pytestmark = pytest.mark.gpu
SHAPES = [(1, 0), (2, 1), (4, 0), (4, 2), (8, 1), (8, 3), (16, 0), (16, 1),
          (16, 2), (16, 3)]


@pytest.fixture(scope="module")
def ctx():
    with Context(0) as c:
        yield c


def scene(name):
    if name.startswith("star"):  # cells of up to that many planes
        n = int(name[4:])
        k = np.arange(n) + 0.5
        ph, th = np.arccos(1 - 2 * k / n), np.pi * (1 + 5 ** 0.5) * k
        d = np.c_[np.cos(th) * np.sin(ph), np.sin(th) * np.sin(ph),
                  np.cos(ph)]
        sph = np.c_[np.r_[[[0.5, 0.48, 0.53]], 0.5 + 0.33 * d],
                    np.full(n + 1, 0.01)]
        return 1, 0.0, sph
    if name == "lattice":  # bisectors through the grid's vertices
        g = (np.arange(4) + 0.5) / 4
        p = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
        return 4, 0.0, np.c_[p, np.full(len(p), 0.05)]
    # coarse tets, many spheres: long chains of cuts, whole facets cut off
    return 2, 0.1, prep.spheres(700, 0, 5, 0.01, 0.15)


@pytest.mark.parametrize("name", ["star9", "star15", "star29", "star45",
                                  "lattice", "dense"])
def test_boundaries_in_every_shape(ctx, name):
    n, jitter, sph = scene(name)
    verts, tets = prep.grid_mesh(n, jitter, 7)
    inst = prep.build_instance(verts, tets, sph)
    orc = oracle.run(inst, mode=0)
    ctx.upload(inst)
    for G, caps in SHAPES:
        ctx.run(cells_per_wave=G, small_caps=caps)
        compare_with_oracle(ctx.download(), orc)
    ctx.run(small_tier=False)
    compare_with_oracle(ctx.download(), orc)
    ctx.run(force_exact=True)
    compare_with_oracle(ctx.download(), orc)
