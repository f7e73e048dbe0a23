"""Renders over a tree deep enough that kernels take more than 64 KB of dynamic LDS: a batch whose
largest request is not its last, and the same frames alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def deep_scene():
    """Overlapping triangles at 28 scales, split down to single ones: 18 levels."""
    rng = np.random.default_rng(0)
    tris = []
    for p in 2.0 ** np.arange(28):
        c = rng.random((30, 3)) * p
        tris.append(np.concatenate([c + rng.normal(size=(30, 3)) * p for _ in range(3)], 1))
    return np.concatenate(tris).astype(np.float32)


def test_batch_over_a_deep_tree(dev):
    import torch
    import dumbray_amd as D
    from dumbray_amd import plugins as PL
    from dumbray_amd import scenes as S
    tris = deep_scene()
    tree = D.Octree(1, 24)
    tree.push(tris)
    scene = tree.build().upload()
    cam = S.Camera.look_at((3e5, 2e5, -4e5), (1e5, 1e5, 1e5))
    mats = [dict(kind="lambert", albedo=(0.7, 0.5, 0.4))]
    lights = [PL.spherical_light((9.0e10, 8.0e10, 7.0e10), (3.0e5, 4.0e5, -2.0e5), 1.0e4)]
    quad = S.spheres_scene(4, seed=1).lights
    shapes = [((4, 4), "spherical_segment", quad), ((17, 16), "stochastic", quad), ((4, 4), "spherical_segment", lights),
              ((17, 16), "stochastic", lights), ((4, 4), "stochastic", quad), ((5, 3), "spherical_segment", lights),
              ((5, 3), "spherical_segment", quad), ((1, 1), "stochastic", lights)]
    rs = [D.DumbRenderer(scene, np.zeros(len(tris), np.int32), mats, l, cam, 9, 7, spp, 1, lens=lens, seed=k,
                         ignore_backfaces=False, lens_params=PL.spherical_segment_lens((70.0, 45.0), 12.0, 0.3, (1.0, 0.8, 0.6)))
          for k, (spp, lens, l) in enumerate(shapes)]
    print(f"[case] batch of {len(rs)} requests over 18 levels", flush=True)
    frames = [D.BlockBasedFrameBuffer(9, 7) for _ in rs]
    batch = D.RenderBatch([(r, f, 1, 0) for r, f in zip(rs, frames)],
                          dict(tile_blocks=1, groups_per_cu=3, refill_min=4))
    for _ in range(2):
        batch.run()
        torch.cuda.synchronize()
        for k, (r, f) in enumerate(zip(rs, frames)):
            assert torch.equal(f.data.view(torch.int32), r.render().data.view(torch.int32)), k
            f.data.zero_()
    g = rs[0]
    ga, ge = g.backward(torch.ones((2 * 128, 4), device="cuda"))
    assert bool(torch.isfinite(ga).all()) and bool(torch.isfinite(ge).all())
