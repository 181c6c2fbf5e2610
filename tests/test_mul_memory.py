"""The multiplicative scheme where the device has no memory for a whole batch of views' work spectra: initialisation goes on
with smaller batches, down to a view a launch, and gives the same values (a view's launches do the same work in any batch).

The allocation fails from the host, MVR_TEST_MAX_VIEW_SPECTRA being the most work spectra it grants.
"""
import numpy as np
import pytest
import torch  # noqa: F401  before the library is loaded: the process then has one HIP runtime, torch's

from mvr import hip
from mvr import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(12, 17, 20), (131, 9, 14)])  # planar spectra, strided passes
@pytest.mark.parametrize("views,granted", [(9, 5), (8, 2), (5, 1), (2, 1)])
def test_smaller_batches_when_memory_is_short(monkeypatch, views, granted, shape):
    w = syn.small_workload(shape=shape, views=views, k=5, psf_type="INDEPENDENT", weights="zramp")
    inp = syn.make_inputs(w)
    d = hip.Decon(shape, views, "INDEPENDENT", "MUL", 6e-4)
    for v in range(views):
        d.set_view(v, inp["imgs"][v], inp["weights"][v], inp["psfs"][v])
    out = []
    for limit in (None, granted, None):  # on one handle: its buffers change size both ways
        if limit:
            monkeypatch.setenv("MVR_TEST_MAX_VIEW_SPECTRA", str(limit))
        else:
            monkeypatch.delenv("MVR_TEST_MAX_VIEW_SPECTRA", raising=False)
        d.init()
        d.run(2)
        out.append(d.psi())
    d.close()
    np.testing.assert_array_equal(out[1], out[0])
    np.testing.assert_array_equal(out[2], out[0])
