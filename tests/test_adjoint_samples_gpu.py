"""Sample counts whose jobs of one framebuffer block no longer fit 31 bits, and those that no 32-bit
sample number can hold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _renderer(spp, size=(3, 2)):
    import dumbray_amd as D
    from dumbray_amd import scenes as S
    sc = S.spheres_scene(4, seed=1)
    tree = D.Octree(16, 12)
    tree.push(sc.tris)
    return D.DumbRenderer(tree.build().upload(), sc.mat_id, sc.materials, sc.lights, sc.camera, *size, spp, 0)


def test_adjoint_of_two_to_the_24_samples(dev):
    """The gradients of 4095 x 4097 and 4096 x 4096 samples a pixel, one sample more, against those of
    2896 x 2896, the last square that one launch takes: estimates from 5 * 10^7 and 10^8 paths, a few 1e-4
    apart at most; a lost part of the jobs would show whole."""
    import torch
    grads = []
    for spp in ((2896, 2896), (4095, 4097), (4096, 4096)):
        g = _renderer(spp)
        print(f"[case] adjoint of 3x2 pixels at {spp} samples", flush=True)
        dl = torch.rand((128, 4), generator=torch.Generator(device="cuda").manual_seed(3), device="cuda")
        ga, ge = g.backward(dl)
        torch.cuda.synchronize()
        grads.append((ga.cpu().numpy(), ge.cpu().numpy()))
    for other in grads[1:]:
        for a, b in zip(grads[0], other):
            assert np.abs(a).max() > 0
            assert np.abs(a - b).max() <= 0.01 * np.abs(a).max()


def test_sample_counts_beyond_31_bits_are_refused(dev):
    import torch
    import dumbray_amd as D
    for spp in ((65536, 65536), (46341, 46341), (2 ** 31 - 1, 2)):
        g = _renderer(spp)
        with pytest.raises(D.DumbRayError):
            g.render()
        with pytest.raises(D.DumbRayError):
            g.backward(torch.zeros((128, 4), device="cuda"))
        with pytest.raises(D.DumbRayError):
            D.RenderBatch([(g, D.BlockBasedFrameBuffer(3, 2), 1, 0)])
