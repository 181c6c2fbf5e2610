"""Second kernels of many views: a view's kernel is normalised when its turn comes, so the products of view v take the kernels
of later views as they were given (DeconViewPSF.init in the order of the views).  The scale decides whether the float32
products stay in range: with sixteen kernels of 729 values, all normalised, they underflow to 0 (and normalise to NaN).

The oracle runs the same order in float32.  Compared are the views whose partial products stay normal numbers, 0 to 8; a
product has 15 factors of up to two convolutions, each within 3e-7 of the oracle's (relative L2): 2e-5.  Kernels of large
values overflow in the first views and are finite in the last, as the oracle's.
"""
import numpy as np
import pytest
import torch  # noqa: F401  before the library is loaded: the process then has one HIP runtime, torch's

from mvr import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("psf_type", ["EFFICIENT_BAYESIAN", "OPTIMIZATION_I"])
@pytest.mark.parametrize("k", [(9, 9, 9), (66, 3, 4)])  # pairs batched, pair by pair
def test_later_kernels_as_given(oracle, psf_type, k):
    V = 16
    ks = np.random.default_rng(sum(k)).uniform(0.01, 1.0, (V,) + k).astype(np.float32)
    k1, k2 = hip.init_psfs(ks, psf_type, 8)
    want1, want2 = oracle.init_psfs(ks, psf_type, 8)
    np.testing.assert_array_equal(k1, want1)
    for v in range(9):
        got, want = k2[v].astype(np.float64), want2[v].astype(np.float64)
        assert np.isfinite(want).all()
        assert np.linalg.norm(got - want) <= 2e-5 * np.linalg.norm(want), v


@pytest.mark.parametrize("psf_type", ["EFFICIENT_BAYESIAN", "OPTIMIZATION_I"])
def test_products_out_of_range(oracle, psf_type):
    V = 4
    ks = (np.random.default_rng(1).uniform(0.5, 1.0, (V, 5, 5, 5)) * 1e20).astype(np.float32)
    _, k2 = hip.init_psfs(ks, psf_type, 8)
    _, want = oracle.init_psfs(ks, psf_type, 8)
    finite = np.isfinite(want)
    assert finite[V - 1].all() and not finite[0].any()
    np.testing.assert_array_equal(np.isfinite(k2), finite)
    assert np.linalg.norm(k2[V - 1] - want[V - 1]) <= 1e-5 * np.linalg.norm(want[V - 1])
