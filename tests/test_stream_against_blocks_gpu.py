"""The streamed frames (k_render_stream) bit for bit against the one-block-per-workgroup kernel
(k_render), at sample counts that both take.  A frame captured in a graph once the scene's work
counters for captured launches are used up runs k_render; the same frame rendered eagerly is streamed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
CAPTURED = 1024                      # kCapturedSlots


@pytest.fixture(scope="module")
def used_up(dev):
    """A scene whose work counters for captured launches are used up."""
    import torch
    import dumbray_amd as D
    from dumbray_amd import scenes as S
    sc = S.spheres_scene(8, seed=0)
    tree = D.Octree(16, 12)
    tree.push(sc.tris)
    scene = tree.build().upload()
    rays = torch.from_numpy(S.primary_rays(sc.camera, 8, 8)).cuda()
    scene.cast(rays)
    torch.cuda.synchronize()
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        for _ in range(CAPTURED):
            scene.cast(rays)
    return sc, scene


@pytest.mark.parametrize("width,height,spp,lens,light", [
    (8, 16, (1, 1), "stochastic", "quad"), (7, 3, (2, 1), "stochastic", "sphere"), (9, 17, (3, 1), "perspective", "quad"),
    (130, 70, (1, 1), "spherical_segment", "quad"), (130, 70, (5, 5), "stochastic", "sphere"),
    (65, 33, (16, 15), "spherical_segment", "quad"), (65, 33, (16, 16), "stochastic", "quad"),
    (33, 18, (16, 16), "stochastic", "sphere"), (257, 129, (3, 3), "stochastic", "quad"), (900, 601, (2, 2), "stochastic", "quad")])
def test_streamed_frame_equals_one_block_per_workgroup(used_up, width, height, spp, lens, light):
    import torch
    import dumbray_amd as D
    from dumbray_amd import plugins as PL
    sc, scene = used_up
    print(f"[case] {width}x{height} spp {spp} {lens} {light}", flush=True)
    lights = sc.lights if light == "quad" else [PL.spherical_light((9.0, 9.0, 9.0), (0.0, 5.0, 0.0), 0.5)]
    g = D.DumbRenderer(scene, sc.mat_id, sc.materials, lights, sc.camera, width, height, spp, 3, lens=lens,
                       lens_params=PL.spherical_segment_lens((70.0, 45.0), 12.0, 0.3, (1.0, 0.8, 0.6)))
    gen = torch.Generator(device="cuda").manual_seed(1)
    for iteration in (1, 3):
        start = torch.rand(D.BlockBasedFrameBuffer(width, height).data.shape, generator=gen, device="cuda")
        frames = [D.BlockBasedFrameBuffer(width, height) for _ in range(3)]
        n = frames[0].getBlockCount()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            g.render(frames[0], iteration)
        for f in frames:
            f.data.copy_(start)
        graph.replay()
        g.render(frames[1], iteration)
        for a in range(0, n, 7):
            g.renderBlocksGPU(frames[2], a, min(n, a + 7), iteration)
        torch.cuda.synchronize()
        bits = [f.data.cpu().numpy().view(np.int32) for f in frames]
        assert not np.array_equal(bits[0], start.cpu().numpy().view(np.int32))
        assert np.array_equal(bits[0], bits[1]) and np.array_equal(bits[0], bits[2]), iteration
