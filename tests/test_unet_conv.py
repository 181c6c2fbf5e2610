"""Network inference at the edges of the convolution kernels' tiles and of what is fused into them.

The convolutions compute 16 x 16 voxel tiles of a plane in columns of planes: one to sixteen planes for one-chunk
inputs through a ring of five planes, four (48 -> 16 channels) or two (32, 64 and 96 input channels) planes otherwise.
The shapes below reach tiles smaller than 16 on every level (4), tiles cut in x and y, columns cut in z and columns
longer than the ring; the view counts reach the input stored with 8 channels (up to seven views) and with 16 (eight).

Tolerance: that of tests/test_unet.py's forward test, rel-L2 <= 2e-3 against the checker that rounds its stored tensors
to bfloat16 as the kernels do (a value near a rounding boundary may round to the other neighbour, 2^-8 relative).
"""
import numpy as np
import pytest

import unet_ref as U

from test_unet import rel


@pytest.mark.gpu
@pytest.mark.parametrize("shape,V", [((4, 4, 4), 7), ((4, 4, 4), 8), ((16, 16, 16), 1), ((12, 36, 20), 8),
                                     ((44, 8, 36), 7), ((30, 33, 17), 6), ((8, 68, 64), 2)])
def test_inference_at_tile_edges(shape, V):
    from mvr import hip
    rng = np.random.default_rng(sum(shape) + V)
    imgs = [rng.uniform(0.0, 4.0, shape).astype(np.float32) for _ in range(V)]
    ws = [rng.uniform(0.0, 1.0, shape).astype(np.float32) for _ in range(V)]
    p = U.random_params(V, seed=V)
    net = hip.UNet(V, seed=0)
    net.set_params(p)
    out = net.infer(imgs, ws, min_value=1e-4)
    net.close()
    ref = U.infer(p, imgs, ws, 1e-4, bf16_mode=True)
    assert out.shape == tuple(shape)
    assert rel(out, ref) <= 2e-3
