"""mvr_fft_convolve_noalloc in a captured graph, the use its header names: small planes transformed beside the kernel's, larger
ones one after the other, and strided passes.

Every replay reads its buffers anew: the image changes between replays, with the program's own work on the scratch array
and synchronisations between them, and each result equals the eager call's bit by bit (the same launches).
"""
import numpy as np
import pytest
import torch

from mvr import hip

pytestmark = pytest.mark.gpu


def convolve(img, k, out, ext, stream):
    hip.fft_convolve_noalloc(img.data_ptr(), tuple(img.shape), k.data_ptr(), tuple(k.shape), out.data_ptr(), ext, 1.0,
                             stream=stream.cuda_stream)


@pytest.mark.parametrize("ext", ["mirror", "value"])
@pytest.mark.parametrize("shape", [(33, 40, 48), (110, 90, 60), (130, 60, 50)])
def test_replays_equal_eager_calls(shape, ext):
    rng = np.random.default_rng(sum(shape))
    imgs = [torch.from_numpy(rng.uniform(0.5, 2.0, shape).astype(np.float32)).cuda() for _ in range(4)]
    k = torch.from_numpy(rng.uniform(0.0, 1.0, (11, 9, 7)).astype(np.float32)).cuda()
    want = torch.empty_like(imgs[0])
    img, out = imgs[0].clone(), torch.full_like(imgs[0], float("nan"))
    torch.cuda.synchronize()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        convolve(img, k, out, ext, stream)
    torch.cuda.synchronize()
    assert torch.isnan(out).all()  # captured, not run
    for other in imgs:
        convolve(other, k, want, ext, stream)
        torch.cuda.synchronize()
        img.copy_(other)
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
