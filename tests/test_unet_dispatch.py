"""Which convolutions the launcher accepts, on the CPU: refusals come before any device work.

launch_conv_tiled is the library's own C++ function, called through its mangled name with an argument block laid out as
ConvArgs of csrc/unet.hpp.
"""
import ctypes
import os

import pytest

from mvr import hip


class PsiArgs(ctypes.Structure):
    _fields_ = [("out", ctypes.c_void_p), ("w", ctypes.c_void_p), ("avg", ctypes.c_void_p), ("scale", ctypes.c_float),
                ("minValue", ctypes.c_float), ("ox", ctypes.c_int), ("oy", ctypes.c_int), ("oz", ctypes.c_int),
                ("zlo", ctypes.c_int)]


class ConvArgs(ctypes.Structure):
    _fields_ = ([("in_", ctypes.c_void_p), ("in_cs", ctypes.c_int), ("cin", ctypes.c_int), ("in_half", ctypes.c_int),
                 ("w", ctypes.c_void_p), ("bias", ctypes.c_void_p), ("out", ctypes.c_void_p), ("out_cs", ctypes.c_int),
                 ("out_co", ctypes.c_int), ("cout", ctypes.c_int)] +
                [(n, ctypes.c_int) for n in ("N", "D", "H", "W", "taps", "relu")] +
                [("up_in", ctypes.c_void_p), ("up_cs", ctypes.c_int), ("up_c", ctypes.c_int),
                 ("pool_out", ctypes.c_void_p), ("pool_cs", ctypes.c_int), ("mask", ctypes.c_void_p),
                 ("mask_cs", ctypes.c_int), ("psi", PsiArgs)])


# (not where a GPU could run what should have been refused)
pytestmark = pytest.mark.skipif(os.path.exists("/dev/kfd"), reason="null operands: for machines without a GPU")


# the kernel of 48 inputs has no backward ReLU, and the others with one take as many outputs as inputs
@pytest.mark.parametrize("cin,cout", [(48, 48), (16, 32), (96, 96), (64, 32)])
def test_backward_relu_without_a_kernel_is_refused(cin, cout):
    launch = getattr(ctypes.CDLL(hip.LIB_PATH), "_ZN3mvr17launch_conv_tiledERKNS_8ConvArgsEP12ihipStream_t")
    launch.argtypes = [ctypes.POINTER(ConvArgs), ctypes.c_void_p]
    launch.restype = ctypes.c_bool
    a = ConvArgs(in_cs=cin, cin=cin, out_cs=cout, cout=cout, N=1, D=4, H=4, W=4, taps=27, mask=16, mask_cs=cout)
    assert not launch(ctypes.byref(a), None)
