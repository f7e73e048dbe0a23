"""A frame buffer's first image conversion works under graph capture as it does eagerly, and what it
forms there is not kept for later calls."""
import pytest

from dumbray_amd.render import BlockBasedFrameBuffer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(1, 1), (8, 16), (37, 21)])
def test_first_conversion_in_a_graph(size):
    import torch

    frame = BlockBasedFrameBuffer(*size)
    gen = torch.Generator(device="cuda").manual_seed(1)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        image = frame.to_image()
        back = frame.from_image(image)
    for _ in range(3):
        frame.data.copy_(torch.rand(frame.data.shape, generator=gen, device="cuda"))
        graph.replay()
        torch.cuda.synchronize()
        eager = frame.to_image()
        assert image.shape == (size[1], size[0], 4)
        assert torch.equal(image, eager)
        assert torch.equal(back, frame.from_image(eager))
        torch.cuda.synchronize()
