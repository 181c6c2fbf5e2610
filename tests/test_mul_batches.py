"""The multiplicative scheme with several views in a launch: more views than a launch holds (8), and grids whose work spectra
fit the bound on a batch (256 MiB) only in parts; planar spectra and strided ones.

Tolerance: iterations within 1e-5 of the checker, as in tests/test_gpu_parity.py; the large grid is compared with the same
iteration put together from single convolutions of the library, 1e-5 likewise.
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


def run(imgs, ws, ks, psf_type, iterations):
    d = hip.Decon(imgs[0].shape, len(imgs), psf_type, "MUL", 6e-4)
    for v in range(len(imgs)):
        d.set_view(v, imgs[v], ws[v], ks[v])
    d.init()
    start = d.psi()
    d.run(iterations)
    psi = d.psi()
    d.close()
    return start, psi


@pytest.mark.parametrize("views", [1, 2, 8, 9, 17])
@pytest.mark.parametrize("shape", [(12, 17, 20), (131, 9, 14)])
def test_views_of_several_launches(oracle, views, shape):
    w = syn.small_workload(shape=shape, views=views, k=5, psf_type="INDEPENDENT", weights="zramp")
    inp = syn.make_inputs(w)
    imgs, ws, ks = inp["imgs"], inp["weights"], inp["psfs"]
    ref = oracle.deconvolve(imgs, ws, ks, psf_type="INDEPENDENT", scheme="MUL", lam=6e-4, iterations=2)
    assert rel(run(imgs, ws, ks, "INDEPENDENT", 2)[1], ref["psi"]) <= 1e-5


def test_batches_cut_by_their_memory():
    # 288 x 240 x 200 points: 59 MB a spectrum, four views to a batch
    shape, V = (190, 230, 282), 5
    rng = np.random.default_rng(3)
    imgs = rng.uniform(0.5, 30.0, (V,) + shape).astype(np.float32)
    ws = rng.uniform(0.1, 0.3, (V,) + shape).astype(np.float32)
    ks = rng.uniform(0.1, 1.0, (V, 5, 7, 5)).astype(np.float32)
    start, psi = run(imgs, ws, ks, "INDEPENDENT", 1)
    k1, k2 = hip.init_psfs(ks, "INDEPENDENT", 8)
    integrals = np.stack([hip.fft_convolve((imgs[v] / hip.fft_convolve(start, k1[v], "mirror", 0.0)).astype(np.float32),
                                           k2[v], "value", 1.0) for v in range(V)])
    want, _ = hip.compute_final_values_mul(start.ravel(), integrals.reshape(V, -1), ws.reshape(V, -1), 6e-4, 1e-4,
                                           float(np.mean([i.max() for i in imgs])))
    assert rel(psi.ravel(), want) <= 1e-5
