"""Grids whose y-z planes are transformed in one pass (FFT lengths up to 128 along y and z and 256 along x), at the
edges of that range and of its rules: the smallest and largest planes, unequal lengths, planes just beyond the range (the
strided passes), volumes of one row or plane, kernels longer than the volume (several reflections at a face), and both
extensions; whole deconvolutions on such grids; batched blocks whose quotient regions are cut by the volume.

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


@pytest.mark.parametrize("shape,k", [((12, 12, 10), (5, 5, 5)), ((1, 9, 14), (3, 3, 3)), ((9, 1, 14), (3, 5, 3)),
                                     ((5, 7, 3), (11, 13, 9)), ((98, 98, 60), (31, 31, 31)), ((120, 14, 226), (9, 3, 31)),
                                     ((99, 98, 60), (31, 31, 31)), ((60, 50, 230), (5, 5, 31)), ((52, 60, 64), (21, 15, 15))])
@pytest.mark.parametrize("ext,value", [("mirror", 0.0), ("value", 0.0), ("value", 1.0)])
def test_convolution(oracle, shape, k, ext, value):
    rng = np.random.default_rng(sum(shape) + sum(k))
    img = rng.uniform(0.5, 2.0, shape).astype(np.float32)
    ker = rng.uniform(0.0, 1.0, k).astype(np.float32)
    ref = oracle.fft_convolve(img.astype(np.float64), ker.astype(np.float64), ext, value, dtype=np.float64)
    assert rel(hip.fft_convolve(img, ker, ext, value), ref) <= 3e-6
    ti, tk = torch.from_numpy(img).cuda(), torch.from_numpy(ker).cuda()
    to = torch.full_like(ti, float("nan"))
    hip.fft_convolve_noalloc(ti.data_ptr(), img.shape, tk.data_ptr(), k, to.data_ptr(), ext, value)
    torch.cuda.synchronize()
    assert rel(to.cpu().numpy(), ref) <= 3e-6


@pytest.mark.parametrize("scheme", ["SEQ", "MUL"])
@pytest.mark.parametrize("shape,k", [((14, 33, 30), 7), ((40, 52, 20), 21), ((98, 20, 36), 31), ((82, 20, 30), 15),
                                     ((86, 20, 30), 15)])
def test_deconvolution(oracle, scheme, shape, k):
    w = syn.small_workload(shape=shape, views=3, k=k, psf_type="EFFICIENT_BAYESIAN", weights="zramp")
    inp = syn.make_inputs(w)
    imgs, ws, ks = inp["imgs"], inp["weights"], inp["psfs"]
    ref = oracle.deconvolve(imgs, ws, ks, psf_type="EFFICIENT_BAYESIAN", scheme=scheme, lam=6e-4, iterations=3)
    d = hip.Decon(shape, 3, "EFFICIENT_BAYESIAN", scheme, 6e-4)
    for v in range(3):
        d.set_view(v, imgs[v], ws[v], ks[v])
    d.init()
    d.run(3)
    psi = d.psi()
    d.close()
    assert rel(psi, ref["psi"]) <= 1e-5


@pytest.mark.parametrize("shape,k,effective", [((40, 30, 52), 9, 16), ((70, 33, 40), 15, 32), ((20, 20, 20), 9, 40)])
def test_batched_blocks_equal_the_frame(shape, k, effective):
    w = syn.small_workload(shape=shape, views=2, k=k, psf_type="OPTIMIZATION_I", weights="zramp")
    inp = syn.make_inputs(w)
    imgs, ws, ks = inp["imgs"], inp["weights"], inp["psfs"]
    out = []
    for block in (0, effective + 2 * (k - 1)):
        d = hip.Decon(shape, 2, "OPTIMIZATION_I", "SEQ", 6e-4)
        for v in range(2):
            d.set_view(v, imgs[v], ws[v], ks[v])
        d.set_block_size((block, block, block))
        d.init()
        d.run(3)
        out.append(d.psi())
        d.close()
    assert rel(out[1], out[0]) <= 1e-5
