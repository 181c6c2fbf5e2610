"""The x passes with a wave's lanes packed with rows: half lengths M = P0/2 of every packing (idle lanes or none, rows at
multiples of 16, 32 or 64 lanes, rows side by side, a sparse or dense second side), odd and even row lengths, fewer rows
than a work-group holds, planar spectra (M <= 128 here) and strided ones (131 rows along y).

Tolerances are those of tests/test_gpu_parity.py: a convolution within 3e-6 of the FP64 checker, iterations within 1e-5.
"""
import numpy as np
import pytest
import torch  # noqa: F401  before the library is loaded: the process then has one HIP runtime, torch's

from mvr import hip
from mvr import synthetic as syn

pytestmark = pytest.mark.gpu


def rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


LENGTHS = [8, 10, 20, 30, 36, 50, 60, 64, 72, 90, 96, 100, 108, 120, 128, 135, 144, 150, 180, 200, 216, 225, 256, 270, 288,
           300, 320, 360, 384, 400, 432, 450, 480, 512, 540, 576, 640]


@pytest.mark.parametrize("odd", [0, 1])
@pytest.mark.parametrize("half", LENGTHS)
def test_convolution(oracle, half, odd):
    for ny in (5, 131):
        img = np.random.default_rng(half + odd).uniform(0.5, 2.0, (2, ny, 2 * half - 4 - odd)).astype(np.float32)
        ker = np.random.default_rng(half).uniform(0.0, 1.0, (3, 3, 5)).astype(np.float32)
        ref = oracle.fft_convolve(img.astype(np.float64), ker.astype(np.float64), "mirror", 0.0, dtype=np.float64)
        assert rel(hip.fft_convolve(img, ker, "mirror", 0.0), ref) <= 3e-6


@pytest.mark.parametrize("odd", [0, 1])
@pytest.mark.parametrize("half", LENGTHS)
def test_iterations(oracle, half, odd):
    for ny in (9, 127):
        shape = (5, ny, 2 * half - 4 - odd)
        w = syn.small_workload(shape=shape, views=2, k=5, psf_type="INDEPENDENT", weights="zramp")
        inp = syn.make_inputs(w)
        imgs, ws, ks = inp["imgs"], inp["weights"], inp["psfs"]
        ref = oracle.deconvolve(imgs, ws, ks, psf_type="INDEPENDENT", scheme="SEQ", lam=6e-4, iterations=2)
        d = hip.Decon(shape, 2, "INDEPENDENT", "SEQ", 6e-4)
        for v in range(2):
            d.set_view(v, imgs[v], ws[v], ks[v])
        d.init()
        d.run(2)
        psi = d.psi()
        d.close()
        assert rel(psi, ref["psi"]) <= 1e-5
