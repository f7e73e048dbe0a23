"""Walks that go on past a held leaf, at the edges of waves and trees: trees of one leaf, of one level
and of many, with leaves that no triangle record fills, and batches of one ray to a few waves.  A ray's
hit does not depend on the others it is cast with, so every batch is the oracle's bit for bit."""
import numpy as np
import pytest

import dumbray_amd as D
from dumbray_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntris,split,depth", [(1, 8, 24), (8, 8, 24), (9, 8, 6), (60, 1, 4), (2000, 1, 3), (2000, 2, 5),
                                               (3000, 5000, 4), (20000, 1, 1)])    # leaves of thousands of records
def test_batches_of_every_size(oracle, ntris, split, depth):
    import torch

    tris = S.random_soup(ntris, seed=ntris, extent=4.0, size=1.0)
    if ntris > 8:
        tris[::7, 3:6] = tris[::7, 0:3]                       # degenerate: in the tree, without a record
    tree = D.Octree(split, depth)
    tree.push(tris)
    tree.build()
    scene = tree.upload()
    want_tree = oracle.Octree(tris, split, depth)
    rng = np.random.default_rng(5)
    cen = tris.reshape(-1, 3, 3).mean(axis=1)
    o = rng.uniform(-6, 6, (1000, 3)).astype(np.float32)
    aim = cen[rng.integers(0, ntris, 1000)]
    d = (aim - o).astype(np.float32)
    d[::5, 0] = 0.0                                           # rays in a coordinate plane
    rays = np.ascontiguousarray(np.concatenate([o, d], 1))
    for clip in (False, True):
        want = want_tree.cast(rays, clip=clip)
        for n in (1, 63, 64, 65, 256, 1000):
            got = scene.cast(torch.from_numpy(rays[:n]).cuda(), clip_backfaces=clip)
            torch.cuda.synchronize()
            assert np.array_equal(got["id"].cpu().numpy(), want["id"][:n])
            hit = want["id"][:n] >= 0
            assert np.array_equal(got["t"].cpu().numpy()[hit].view(np.int32), want["t"][:n][hit].view(np.int32))
