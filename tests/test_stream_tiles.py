"""A host model of k_render_stream's job stream (dumbray_amd/csrc/dr_render.hip): tiles fetched in
stream order into a ring of ids, each wave's queue of `chunk` prepared jobs, the ring of pixel slots
that gates a job's start, and the end of the stream.  Waves run one loop iteration at a time in
random order and paths take random numbers of iterations, a few of them very many.  Every run must
end, every pixel of every tile must be written once from all of its samples, and no ring entry or
slot may be reused while a job still needs it.

On the GPU: frames of every size class and sample count equal the one-block-per-workgroup kernel's
(RenderBatch) bit for bit, also through ranges of blocks and when blended."""
import random

import numpy as np
import pytest

RING, SAMPLES, SHADE_MIN, REFILL_MIN = 64, 2048, 32, 4


def slots_of(spp):
    n = 1
    while 2 * n * spp <= SAMPLES:
        n *= 2
    return 0 if spp == 1 else n


def stream(seed, ntiles, tile, spp, chunk, nwg, waves=4, ring=RING, maxlen=12, long_p=0.0, long_len=0):
    rnd = random.Random(seed)
    assert tile * spp % chunk == 0
    nslots = slots_of(spp)
    fetched, written = 0, {}
    wgs = [dict(owner=list(range(nslots)), remaining=[spp] * nslots, staged={}, tiles=[None] * ring, done=[0] * ring,
                next=0, end=1 << 30, left=waves,
                waves=[dict(base=0, pos=0, len=0, taken=False, ended=False, over=False, lanes=[None] * 64)
                       for _ in range(waves)]) for _ in range(nwg)]

    def pixel_written(wg, u, samples):
        k = u // tile
        n, tid = wg["tiles"][k % ring]
        assert n == k, "ring entry reused while a pixel of its tile was open"
        key = (tid, u % tile)
        assert key not in written and samples == list(range(spp))
        written[key] = True
        wg["done"][k % ring] += 1

    def iteration(wg, wv):
        nonlocal fetched
        lanes = wv["lanes"]
        live = [i for i in range(64) if lanes[i]]
        done = [i for i in live if lanes[i][2] == 0]
        if done and len(done) * 64 >= len(live) * SHADE_MIN:
            for i in done:
                u, s, _ = lanes[i]
                lanes[i] = None
                if nslots == 0:
                    pixel_written(wg, u, [s])
                    continue
                slot = u % nslots
                assert wg["owner"][slot] == u, "slot reused while a job of its pixel ran"
                wg["staged"].setdefault(slot, []).append(s)
                wg["remaining"][slot] -= 1
                if wg["remaining"][slot] == 0:
                    wg["remaining"][slot] = spp
                    pixel_written(wg, u, sorted(wg["staged"].pop(slot)))
                    wg["owner"][slot] = u + nslots
        if wv["pos"] == wv["len"] and not wv["ended"]:
            if not wv["taken"]:
                wv["base"], wg["next"], wv["taken"] = wg["next"], wg["next"] + chunk, True
            k = wv["base"] // spp // tile
            past, entry = k >= wg["end"], None
            if not past and wg["done"][k % ring] >= (k // ring) * tile:
                entry = wg["tiles"][k % ring]
                if entry is not None and entry[0] != k:
                    entry = None
                if entry is None and wv["base"] == k * tile * spp:
                    prev = wg["tiles"][(k - 1) % ring]
                    if k == 0 or (prev is not None and prev[0] == k - 1):
                        if fetched >= ntiles:
                            wg["end"], past = min(wg["end"], k), True
                        else:
                            entry = wg["tiles"][k % ring] = (k, fetched)
                        fetched += 1
            wv["ended"] = past
            if entry is not None:
                wv["taken"], wv["pos"], wv["len"] = False, 0, chunk
        idle = [i for i in range(64) if not lanes[i]]
        if wv["pos"] < wv["len"] and (len(idle) >= REFILL_MIN or len(idle) == 64):
            for i in idle:
                if wv["pos"] == wv["len"]:
                    break
                u, s = divmod(wv["base"] + wv["pos"], spp)
                if nslots and wg["owner"][u % nslots] != u:
                    break
                dur = long_len if rnd.random() < long_p else rnd.randint(0, maxlen)
                lanes[i] = [u, s, dur]
                wv["pos"] += 1
        if not any(lanes):
            if wv["pos"] == wv["len"] and wv["ended"]:
                wv["over"] = True
            return
        for x in lanes:
            if x and x[2] > 0:
                x[2] -= 1

    steps = 0
    while any(not wv["over"] for wg in wgs for wv in wg["waves"]):
        wg = rnd.choice(wgs)
        wv = rnd.choice(wg["waves"])
        if not wv["over"]:
            iteration(wg, wv)
        steps += 1
        assert steps < 400000, "the stream stalls"
    assert len(written) == ntiles * tile


@pytest.mark.parametrize("ntiles,tile,spp,chunk,nwg", [
    (1, 128, 1, 8, 1), (7, 64, 1, 64, 2), (300, 8, 9, 8, 2), (40, 16, 4, 64, 3), (12, 128, 16, 64, 2), (5, 8, 255, 8, 1),
    (200, 8, 8, 8, 1), (3, 64, 3, 64, 4)])
@pytest.mark.parametrize("long_p", [0.0, 0.02])
def test_stream_ends_and_writes_every_pixel_once(ntiles, tile, spp, chunk, nwg, long_p):
    for seed in range(2):
        stream(seed, ntiles, tile, spp, chunk, nwg, long_p=long_p, long_len=400)


@pytest.mark.gpu
@pytest.mark.parametrize("width,height,spp,lens", [
    (8, 16, (1, 1), "stochastic"), (7, 3, (2, 1), "stochastic"), (9, 17, (3, 1), "perspective"),
    (130, 70, (1, 1), "spherical_segment"), (130, 70, (5, 5), "stochastic"), (64, 33, (16, 16), "stochastic"),
    (64, 33, (16, 15), "spherical_segment"), (257, 129, (3, 3), "stochastic")])
def test_streamed_frame_equals_one_block_kernel(dev, width, height, spp, lens):
    import torch
    import dumbray_amd as D
    from dumbray_amd import plugins as PL
    from dumbray_amd import scenes as S
    print(f"[case] stream {width}x{height} spp {spp} {lens}", flush=True)
    sc = S.spheres_scene(8, seed=0)
    tree = D.Octree(16, 12)
    tree.push(sc.tris)
    g = D.DumbRenderer(tree.build().upload(), sc.mat_id, sc.materials, sc.lights, sc.camera, width, height, spp, 3,
                       lens=lens, lens_params=PL.spherical_segment_lens((70.0, 45.0), 12.0, 0.3, (1.0, 0.8, 0.6)))
    gen = torch.Generator(device="cuda").manual_seed(1)
    for iteration in (1, 3):
        start = torch.rand(D.BlockBasedFrameBuffer(width, height).data.shape, generator=gen, device="cuda")
        frames = [D.BlockBasedFrameBuffer(width, height) for _ in range(3)]
        for f in frames:
            f.data.copy_(start)
        g.render(frames[0], iteration)
        n = frames[1].getBlockCount()
        for a in range(0, n, 5):
            g.renderBlocksGPU(frames[1], a, min(n, a + 5), iteration)
        D.RenderBatch([(g, frames[2], iteration, 0)], dict(tile_blocks=2, groups_per_cu=1, refill_min=8)).run()
        torch.cuda.synchronize()
        bits = [f.data.cpu().numpy().view(np.int32) for f in frames]
        assert np.array_equal(bits[0], bits[1]) and np.array_equal(bits[0], bits[2]), iteration


@pytest.mark.gpu
@pytest.mark.parametrize("tuning", [None, dict(tile_blocks=3, groups_per_cu=1, refill_min=16),
                                    dict(tile_blocks=1, groups_per_cu=4, refill_min=1)])
def test_batch_of_streams_and_rounds(dev, tuning):
    """One batch with streamed requests of every slot count, requests above the streamed kernel's 256
    samples a pixel, and more requests than one wave looks over: each frame is its solo frame."""
    import torch
    import dumbray_amd as D
    from dumbray_amd import plugins as PL
    from dumbray_amd import scenes as S
    sc = S.spheres_scene(4, seed=1)
    tree = D.Octree(16, 12)
    tree.push(sc.tris)
    scene = tree.build().upload()
    shapes = [(40, 24, (1, 1)), (24, 40, (17, 16)), (33, 17, (16, 16)), (130, 70, (2, 1)), (8, 16, (20, 20))]
    shapes += [(8 + k % 5, 16 + k % 3, (1 + k % 3, 1)) for k in range(70)]
    rs = [D.DumbRenderer(scene, sc.mat_id, sc.materials, sc.lights if k % 4 else [PL.spherical_light((9.0, 9.0, 9.0), (0.0, 5.0, 0.0), 0.5)],
                         sc.camera, w, h, spp, 2, seed=k) for k, (w, h, spp) in enumerate(shapes)]
    print(f"[case] batch of {len(rs)} streams and rounds, {tuning}", flush=True)
    frames = [D.BlockBasedFrameBuffer(r.width, r.height) for r in rs]
    batch = D.RenderBatch([(r, f, 1, 0) for r, f in zip(rs, frames)], tuning)
    for replay in range(3):
        for f in frames:
            f.data.zero_()
        batch.run()
        torch.cuda.synchronize()
        for k, (r, f) in enumerate(zip(rs, frames)):
            assert torch.equal(f.data.view(torch.int32), r.render().data.view(torch.int32)), (replay, k)
