"""Second kernels of several views: all pairs of views batched on grids transformed plane by plane, one pair at a time on
larger ones (FFT lengths above 128 along y or z, 256 along x), against the same chains of single convolutions.

Sizes: two views up to more than one batch holds (seven 61^3 kernels: 56 MB of pairs per view, 256 MB a batch), even and
single extents, the sizes on both sides of the larger grids.

Tolerance: the chains run the same transforms and products in float32, so only the order within a transform could differ:
1e-6 (relative L2) is 8 float32 roundings for chains of up to 12 convolutions.
"""
import numpy as np
import pytest
import torch  # noqa: F401  before the library is loaded: the process then has one HIP runtime, torch's

from mvr import hip

pytestmark = pytest.mark.gpu


def mirrored(a):
    for axis, n in enumerate(a.shape):
        idx = np.arange(n)
        for i in range(n // 2 + 1):
            if i < n:
                idx[i], idx[n - 1 - i] = idx[n - 1 - i], idx[i]
        a = np.take(a, idx, axis)
    return np.ascontiguousarray(a)


def chain(ks, psf_type):
    out = []
    inv = [mirrored(k) for k in ks]
    for v in range(len(ks)):
        tmp = inv[v] if psf_type == "EFFICIENT_BAYESIAN" else ks[v]
        for w in range(len(ks)):
            if w == v:
                continue
            if psf_type == "EFFICIENT_BAYESIAN":
                o = hip.fft_convolve(hip.fft_convolve(inv[v], ks[w], "value", 0.0), inv[w], "value", 0.0)
            else:
                o = hip.fft_convolve(ks[v], inv[w], "value", 0.0)
            tmp = o * tmp
        out.append(tmp if psf_type == "EFFICIENT_BAYESIAN" else mirrored(tmp))
    return out


@pytest.mark.parametrize("psf_type", ["EFFICIENT_BAYESIAN", "OPTIMIZATION_I"])
@pytest.mark.parametrize("views,k", [(2, (1, 1, 1)), (3, (5, 8, 1)), (6, (12, 9, 10)), (7, (61, 61, 61)), (3, (64, 4, 6)),
                                     (3, (65, 4, 6)), (2, (6, 66, 7)), (2, (5, 3, 130))])
def test_products_equal_the_chains(views, k, psf_type):
    rng = np.random.default_rng(sum(k) + views)
    ks = rng.uniform(0.2, 1.0, (views,) + k).astype(np.float32)
    k1, k2 = hip.init_psfs(ks, psf_type, 8)
    for got, want in zip(k2, chain(list(k1), psf_type)):
        got = np.asarray(got, np.float64)
        want = np.asarray(want, np.float64)
        got, want = got / got.sum(), want / want.sum()
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)
