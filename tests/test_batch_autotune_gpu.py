"""RenderBatch without a tuning: the autotuner's proxy launches leave the request frames alone, its choice
is a launch shape that a caller could give, and frames are the solo frames."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [
    [((8, 16), (1, 1))], [((40, 24), (2, 2)), ((130, 70), (1, 1))], [((24, 33), (17, 16))],
    [((200, 100), (4, 4)), ((24, 33), (20, 20)), ((500, 300), (3, 3)), ((7, 5), (16, 16))]])
def test_tuned_batch(dev, shapes):
    import torch
    import dumbray_amd as D
    from dumbray_amd import plugins as PL
    from dumbray_amd import scenes as S
    sc = S.spheres_scene(4, seed=1)
    tree = D.Octree(16, 12)
    tree.push(sc.tris)
    scene = tree.build().upload()
    sphere = [PL.spherical_light((9.0, 9.0, 9.0), (0.0, 5.0, 0.0), 0.5)]
    rs = [D.DumbRenderer(scene, sc.mat_id, sc.materials, sc.lights if k % 2 == 0 else sphere, sc.camera, w, h, spp, 2,
                         seed=k) for k, ((w, h), spp) in enumerate(shapes)]
    print(f"[case] autotuned batch of {shapes}", flush=True)
    for iteration in (1, 3):
        frames = [D.BlockBasedFrameBuffer(r.width, r.height) for r in rs]
        want = [D.BlockBasedFrameBuffer(r.width, r.height) for r in rs]
        for k, (f, s) in enumerate(zip(frames, want)):
            f.data.fill_(0.25 + k)
            s.data.fill_(0.25 + k)
        batch = D.RenderBatch([(r, f, iteration, 0) for r, f in zip(rs, frames)])
        torch.cuda.synchronize()
        assert all(bool((f.data == 0.25 + k).all()) for k, f in enumerate(frames))
        t = batch.tuning
        queued = any(x * y > 256 for _, (x, y) in shapes)
        assert t["groups_per_cu"] in (2, 3, 4) and t["refill_min"] in (1, 4, 8)
        assert t["tile_blocks"] in ((1, 2, 4) if queued else (1,))
        batch.run()
        for r, s in zip(rs, want):
            r.render(s, iteration)
        torch.cuda.synchronize()
        for f, s in zip(frames, want):
            assert torch.equal(f.data.view(torch.int32), s.data.view(torch.int32))
