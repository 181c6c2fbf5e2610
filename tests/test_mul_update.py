"""The multiplicative update and the average initial estimate over every number of views up to 32 (their kernels take the
views in fours, and up to 4, 8, 16 and 32), products at the ends of the double range, and values of no root.

Tolerances: the update's root is good to a few roundings of a double, so its float differs from the checker's by at most
the last place, and seldom (as in tests/test_methods.py); maxima are exact and the average is of float inputs in double.
"""
import numpy as np
import pytest
import torch  # noqa: F401  before the library is loaded: the process then has one HIP runtime, torch's

from mvr import hip
from mvr import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [1, 2, 3, 4, 5, 8, 9, 16, 31, 32])
@pytest.mark.parametrize("scale", [1e-36, 1.0, 1e36])
def test_final_values(oracle, V, scale):
    rng = np.random.default_rng(V)
    n = 30011
    last = rng.uniform(1e-4, 500.0, n).astype(np.float32)
    integ = (rng.uniform(0.3, 3.0, (V, n)) * scale).astype(np.float32)
    integ[0, ::31] = 0.0
    integ[-1, 5::97] = np.inf
    integ[0, 7::101] = np.nan
    integ[-1, 11::103] *= -1
    w = rng.uniform(0.0, 0.6, (V, n)).astype(np.float32)
    got, _ = hip.compute_final_values_mul(last, integ, w, 6e-4, 1e-4, 250.0)
    want, _ = oracle.compute_final_values_mul(last, integ, w, 6e-4, 1e-4, 250.0)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    diff = np.abs(got[ok].view(np.int32).astype(np.int64) - want[ok].view(np.int32).astype(np.int64))
    assert diff.max() <= 1 and np.count_nonzero(diff) <= n // 1000


@pytest.mark.parametrize("V", [1, 4, 5, 8, 9, 17])
@pytest.mark.parametrize("shape", [(1, 1, 3), (33, 95, 171)])
def test_average(V, shape):
    rng = np.random.default_rng(V)
    imgs = rng.uniform(-0.5, 2.0, (V,) + shape).astype(np.float32)
    d = hip.Decon(shape, V, "INDEPENDENT", "SEQ", 6e-4)
    for v in range(V):
        d.set_view(v, imgs[v], np.ones(shape, np.float32), syn.gaussian_psf(3, 1.0, 1.0, 0))
    d.init()
    psi = d.psi()
    d.close()
    pos = imgs.astype(np.float64) * (imgs > 0)
    c = (imgs > 0).sum(0)
    avg = (pos.sum(0)[c > 0] / c[c > 0]).mean()
    np.testing.assert_allclose(psi, np.float32(avg), rtol=1e-7 * 2)
