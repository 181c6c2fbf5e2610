"""Weight and bias gradients of the 3^3 layers at the edges of the gradient kernel's tiles.

A patch of P voxels runs its layers at widths P, P/2 and P/4; the kernel tiles a plane into 32 x 4, 16 x 8 or 8 x 16
voxels, whichever pads it least, and deals the tiles over partitions of at least two.  The patches below reach one
partial tile (4, 12), one tile per plane, rows and columns of partial tiles (20, 36, 40), every tile shape, one
partition and many, and one to three samples.

Tolerances: those of tests/test_unet.py, against the checker that rounds its stored tensors to bfloat16 as the kernels
do: an activation or gradient whose FP32 value lies near a rounding boundary may round to the other neighbour (2^-8
relative) in all layers before it, which the bars of 2e-2 relative and 0.999 cosine per layer cover; the last layer's
gradients have only the forward pass before them.
"""
import numpy as np
import pytest

import unet_ref as U

from test_unet import _oracle_batch, _train_problem, rel


@pytest.mark.gpu
@pytest.mark.parametrize("P,batch", [(4, 1), (8, 3), (12, 1), (20, 2), (32, 1), (36, 1), (40, 1)])
def test_weight_gradients_at_tile_edges(P, batch):
    from mvr import hip
    V = 2
    vols = _train_problem(V, P + 4, 2, 100 + P)
    net = hip.UNet(V, seed=0)
    p = U.random_params(V, seed=200 + P)
    net.set_params(p)
    for imgs, ws, tgt in vols:
        net.add_volume(imgs, ws, tgt)
    vidx = [b % 2 for b in range(batch)]
    origins = [(b % 5, (2 * b + 1) % 5, 4 - b) for b in range(batch)]
    net.train_step(vidx, origins, P, lr=0.0, update=False)
    g = net.grads()
    net.close()
    x0, avg, tg = _oracle_batch(vols, vidx, origins, P)
    _, ref = U.loss_and_grads(p, x0, avg, tg, bf16_mode=True)
    at = 0
    for l in range(10):
        for what, n in (("weights", 27 * U.COUT[l] * U.CIN[l]), ("bias", U.COUT[l])):
            a, b = g[at:at + n].astype(np.float64), ref[at:at + n]
            at += n
            cos = float(np.dot(a, b) / (np.linalg.norm(a) * np.linalg.norm(b)))
            assert rel(a, b) <= 2e-2 and cos >= 0.999, f"layer {l} {what}: rel {rel(a, b):.2e} cos {cos:.6f}"
