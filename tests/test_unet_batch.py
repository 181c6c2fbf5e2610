"""Training batches on both sides of a launch's eight patches, of patches from different volumes and origins.

Tolerances: a batch's loss is the mean of its patches' losses, the same float values summed in double (1e-6); its gradient is
the mean of theirs up to the bfloat16 rounding of the stored gradients (the bars of tests/test_unet.py).
"""
import numpy as np
import pytest

from test_unet import _train_problem, rel
import unet_ref as U


@pytest.mark.gpu
@pytest.mark.parametrize("V,batch", [(1, 1), (3, 8), (8, 9), (2, 17)])
def test_batch_is_the_mean_of_its_patches(V, batch):
    from mvr import hip
    P = 8
    net = hip.UNet(V, seed=0)
    net.set_params(U.random_params(V, seed=V))
    for imgs, ws, tgt in _train_problem(V, P + 4, 3, 7 + V):
        net.add_volume(imgs, ws, tgt)
    vidx = [b % 3 for b in range(batch)]
    origins = [(b % 5, (2 * b + 1) % 5, (3 * b) % 4) for b in range(batch)]
    loss = net.train_step(vidx, origins, P, lr=0.0, update=False)
    g = net.grads().astype(np.float64)
    losses, grads = [], []
    for v, o in zip(vidx, origins):
        losses.append(net.train_step([v], [o], P, lr=0.0, update=False))
        grads.append(net.grads().astype(np.float64))
    net.close()
    assert loss == pytest.approx(np.mean(losses), rel=1e-6)
    mean = np.mean(grads, axis=0)
    cos = float(np.dot(g, mean) / (np.linalg.norm(g) * np.linalg.norm(mean)))
    assert rel(g, mean) <= 2e-2 and cos >= 0.999
