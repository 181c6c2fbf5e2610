"""Training steps of callers that do not ask for the loss: the C entry point takes a null pointer for it.

Both networks run the same launches on the same values, so parameters and gradients are equal bit by bit.
"""
import ctypes

import numpy as np
import pytest

from test_unet import _train_problem
import unet_ref as U


@pytest.mark.gpu
@pytest.mark.parametrize("update", [0, 1])
def test_step_without_the_loss(update):
    from mvr import hip
    V, P = 2, 8
    imgs, ws, tgt = _train_problem(V, P + 4, 1, 5)[0]
    vidx, origin = (ctypes.c_int * 1)(0), (ctypes.c_int * 3)(1, 2, 3)
    out = []
    for loss in (ctypes.byref(ctypes.c_double()), None):
        net = hip.UNet(V, seed=0)
        net.set_params(U.random_params(V, seed=1))
        net.add_volume(imgs, ws, tgt)
        rc = hip.lib().mvr_unet_train_step(net.h, vidx, origin, 1, P, 1e-3, update, loss)
        out.append((rc, net.grads(), net.params()))
        net.close()
    assert [rc for rc, _, _ in out] == [0, 0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
    np.testing.assert_array_equal(out[0][2], out[1][2])
    assert np.abs(out[1][1]).max() > 0
