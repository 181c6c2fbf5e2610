"""Convolutions whose passes transform only the rows that hold source values: constant rows of an extension by a value and
the zero rows around a kernel are put in by the pass that reads them.  Even and single-row kernels, kernels as long as the
grid, on grids transformed plane by plane and on grids with strided passes.

Tolerance: a convolution within 3e-6 of the FP64 checker (relative L2), as in tests/test_gpu_parity.py.
"""
import numpy as np
import pytest
import torch  # noqa: F401  before the library is loaded: the process then has one HIP runtime, torch's

from mvr import hip

pytestmark = pytest.mark.gpu


def rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# (130, 7, 9) to (12, 9, 260) have strided passes: 135 and 144 points along y or z, 288 along x; after them planes of 64
# and 96 points, whose kernel's plane is transformed beside the data's, and of 100, whose kernel's plane goes first
@pytest.mark.parametrize("shape,k", [((9, 10, 11), (1, 1, 1)), ((13, 6, 17), (4, 6, 2)), ((1, 5, 8), (8, 1, 12)),
                                     ((1, 1, 2), (16, 16, 16)), ((130, 7, 9), (4, 1, 6)), ((6, 131, 20), (3, 12, 4)),
                                     ((12, 9, 260), (10, 7, 20)), ((48, 50, 12), (17, 15, 5)),
                                     ((80, 82, 20), (15, 15, 9)), ((50, 80, 20), (15, 17, 9)), ((86, 50, 12), (15, 15, 5))])
@pytest.mark.parametrize("ext,value", [("mirror", 0.0), ("value", 0.0), ("value", -2.5)])
def test_convolution(oracle, shape, k, ext, value):
    rng = np.random.default_rng(sum(shape) * 31 + sum(k))
    img = rng.uniform(0.5, 2.0, shape).astype(np.float32)
    ker = rng.uniform(0.0, 1.0, k).astype(np.float32)
    ref = oracle.fft_convolve(img.astype(np.float64), ker.astype(np.float64), ext, value, dtype=np.float64)
    assert rel(hip.fft_convolve(img, ker, ext, value), ref) <= 3e-6
    ti, tk = torch.from_numpy(img).cuda(), torch.from_numpy(ker).cuda()
    to = torch.full_like(ti, float("nan"))
    hip.fft_convolve_noalloc(ti.data_ptr(), img.shape, tk.data_ptr(), k, to.data_ptr(), ext, value)
    torch.cuda.synchronize()
    assert rel(to.cpu().numpy(), ref) <= 3e-6


@pytest.mark.parametrize("shape", [(20, 20, 20), (140, 9, 10)])
def test_value_that_is_not_a_number(shape):
    img = np.ones(shape, np.float32)
    assert np.isnan(hip.fft_convolve(img, np.ones((3, 3, 3), np.float32), "value", float("nan"))).all()
