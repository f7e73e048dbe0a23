"""The adjoint's three forms of workgroup sums (k_backward<kSums...>), chosen by the size of the
material table: the gradients of a table padded until each form is taken are the oracle's FP64 ones,
within the bound of the other adjoint tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LDS, WAVES = 160 * 1024, 4
QUEUES, LEAF = WAVES * 64 * 11 * 4, WAVES * (64 * 8 + 64)


def _form(stacks, n):
    """The rule of backward_shape for n materials and lights."""
    fixed = stacks + QUEUES + LEAF
    per_cu = lambda width: min(3, LDS // (fixed + 3 * n * width))
    if per_cu(8) > 0 and per_cu(8) >= per_cu(4):
        return "fp64"
    return "fp32" if per_cu(4) > 0 else "tight"


@pytest.mark.parametrize("spp", [(1, 1), (2, 2), (6, 5)])
@pytest.mark.parametrize("lens", ["stochastic", "spherical_segment"])
def test_gradients_of_padded_material_tables(dev, oracle, spp, lens):
    import torch
    import dumbray_amd as D
    from dumbray_amd import plugins as PL
    from dumbray_amd import scenes as S
    from test_cast_gpu import _reached_depth
    W, H, depth = 70, 53, 3
    sc = S.spheres_scene(8, seed=0, n_lights=2)
    nl = len(sc.lights)
    lens_params = PL.spherical_segment_lens((70.0, 45.0), 12.0, 0.3, (1.0, 0.8, 0.6))
    kw = dict(lens=PL.STOCHASTIC_LENS if lens == "stochastic" else PL.SPHERICAL_SEGMENT_LENS, lens_params=lens_params)
    o = oracle.Renderer(oracle.Octree(sc.tris, 16, 12), sc.mat_id, sc.materials, sc.lights, sc.camera.as_array(), W, H,
                        spp, depth, **kw)
    w = np.random.default_rng(1).uniform(-1, 1, (H, W, 3)).astype(np.float32)
    oa, oe = o.backward(w)
    tree = D.Octree(16, 12)
    tree.push(sc.tris)
    scene = tree.build().upload()
    stacks = _reached_depth(sc.tris, 16, 12) * 2048
    most = (LDS - stacks) // 12 - nl                       # the largest table that is not refused
    wanted = {}
    for n in list(range(len(sc.materials), most, 50)) + [most - 190, most]:
        wanted.setdefault(_form(stacks, n + nl), []).append(n)
    assert set(wanted) == {"fp64", "fp32", "tight"}
    sizes = [(f, n) for f, ns in wanted.items() for n in {ns[0], ns[-1]}]
    for form, n in sizes:
        print(f"[case] adjoint {W}x{H} spp {spp} {lens}, {n} materials: {form}", flush=True)
        # the scene's materials at the end of the table and its first one, unused ones between
        shift = n - len(sc.materials)
        mats = [sc.materials[0]] * shift + list(sc.materials)
        g = D.DumbRenderer(scene, sc.mat_id + shift, mats, sc.lights, sc.camera, W, H, spp, depth, **kw)
        if n == most:                                      # ... and the first parameters in use too
            g = D.DumbRenderer(scene, np.where(sc.mat_id == 0, 0, sc.mat_id + shift), mats, sc.lights, sc.camera, W, H,
                               spp, depth, **kw)
        dl = D.BlockBasedFrameBuffer(W, H).from_image(torch.from_numpy(w).cuda())
        ga, ge = g.backward(dl)
        torch.cuda.synchronize()
        ga, ge = ga.cpu().numpy(), ge.cpu().numpy()
        got = ga[shift:].copy()
        if n == most and shift:
            got[0] += ga[0]
            ga[0] = 0.0
        assert not ga[:shift].any()
        assert np.all(np.abs(got - oa) <= 1e-4 * np.abs(oa) + 1e-6 * np.abs(oa).max()), (form, n)
        assert np.all(np.abs(ge - oe) <= 1e-4 * np.abs(oe) + 1e-9), (form, n)
    with pytest.raises(D.DumbRayError):
        n = most + 1
        D.DumbRenderer(scene, sc.mat_id, [sc.materials[0]] * n, sc.lights, sc.camera, W, H, spp, depth).backward(dl)
