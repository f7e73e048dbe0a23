"""Work counters of launches under graph capture: a captured launch shares its pair with no other
launch, since it may be replayed beside any of them; once the pairs for captured launches are used up,
a captured frame takes the kernel that needs none."""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CAPTURED, EAGER = 1024, 16384        # kCapturedSlots, kEagerSlots


def test_slots_of_captured_launches_are_their_own(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "probe")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I" + os.path.join(HERE, "..", "dumbray_amd", "csrc"),
                    os.path.join(HERE, "cpp", "work_slots_probe.cpp"), "-o", exe], check=True)
    assert subprocess.run([exe], capture_output=True, text=True, timeout=60).stdout == "ok\n"


@pytest.mark.gpu
def test_eager_slots_are_used_again(dev):
    """More eager casts than there are pairs in the ring: the last of them and a frame are the first's."""
    import torch
    import dumbray_amd as D
    from dumbray_amd import scenes as S
    sc = S.spheres_scene(4, seed=1)
    tree = D.Octree(16, 12)
    tree.push(sc.tris)
    scene = tree.build().upload()
    g = D.DumbRenderer(scene, sc.mat_id, sc.materials, sc.lights, sc.camera, 20, 18, (2, 2), 2)
    rays = torch.from_numpy(S.primary_rays(sc.camera, 8, 8)).cuda()
    frame, first = g.render().data, scene.cast(rays)["id"]
    print(f"[case] {EAGER} eager casts", flush=True)
    for k in range(EAGER + 8):
        out = scene.cast(rays)
        if k % 1024 == 0 or k >= EAGER - 8:
            assert torch.equal(out["id"], first), k
    assert torch.equal(g.render().data.view(torch.int32), frame.view(torch.int32))


@pytest.mark.gpu
def test_captured_frames_beside_eager_launches(dev):
    """More captured frames and casts than there are pairs for them, replayed between eager launches."""
    import torch
    import dumbray_amd as D
    from dumbray_amd import scenes as S
    sc = S.spheres_scene(4, seed=1)
    tree = D.Octree(16, 12)
    tree.push(sc.tris)
    scene = tree.build().upload()
    g = D.DumbRenderer(scene, sc.mat_id, sc.materials, sc.lights, sc.camera, 20, 18, (2, 2), 2)
    rays = torch.from_numpy(S.primary_rays(sc.camera, 16, 16)).cuda()
    eager = g.render().data.clone()
    ids = scene.cast(rays)["id"].clone()
    torch.cuda.synchronize()
    graphs = []
    for n in (1, CAPTURED, 3):
        print(f"[case] graph of {n} casts and 2 frames", flush=True)
        first, last = D.BlockBasedFrameBuffer(20, 18), D.BlockBasedFrameBuffer(20, 18)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            g.render(first)
            for _ in range(n):
                out = scene.cast(rays)
            g.render(last)
        graphs.append((graph, first, last, out))
    for _ in range(3):
        for graph, first, last, out in graphs:
            first.data.zero_()
            last.data.zero_()
            graph.replay()
            again = g.render().data
            torch.cuda.synchronize()
            assert torch.equal(out["id"], ids)
            for data in (first.data, last.data, again):
                assert np.array_equal(data.cpu().numpy().view(np.int32), eager.cpu().numpy().view(np.int32))
