"""Input preparation on device memory, which the kernels read and write in place, against the same calls on host arrays
(staged through the library's own buffers): the same kernels on the same values, so the results are equal bit for bit.
Covered: every entry point with device arrays, an output that overlaps an input (such calls are staged as a whole),
groups of one view, of as many as the kernel arguments hold and of more, blending weights inside, at and beyond their
ranges, equal and different blendings, and widths around a work-group's 256 voxels.
"""
import ctypes

import numpy as np
import pytest
import torch  # before the library is loaded: the process then has one HIP runtime, torch's

pytestmark = pytest.mark.gpu

AFFINE = np.array([[0.96, 0.10, -0.05, 2.5], [-0.08, 1.02, 0.04, 1.25], [0.03, -0.06, 0.98, 3.0]])


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _call(name, *args):
    from mvr import hip
    rc = getattr(hip.lib(), name)(*args)
    assert rc == 0, hip.lib().mvr_last_error().decode()


def _box(shape):
    return (ctypes.c_int * 3)(shape[2], shape[1], shape[0])


def _aff(a=AFFINE):
    return np.ascontiguousarray(a, np.float64).ctypes.data_as(ctypes.POINTER(ctypes.c_double))


BB = (ctypes.c_longlong * 3)(-1, 2, 0)


@pytest.mark.parametrize("out", [(9, 11, 255), (5, 6, 257)])
def test_transforms_on_device_memory(out):
    from mvr import hip
    img = np.random.default_rng(1).uniform(0, 9, (14, 16, 250)).astype(np.float32)
    t, o = _dev(img), torch.full(out, float("nan"), device="cuda")
    _call("mvr_transform_view", 0, _p(t), _box(img.shape), _aff(), BB, _box(out), 1, 1.0, 0.0, 1, _p(o))
    assert np.array_equal(o.cpu().numpy(), hip.transform_view(img, AFFINE, tuple(BB), out))
    bo, bl = (ctypes.c_float * 3)(1.5, 0.0, 1.0), (ctypes.c_float * 3)(6.0, 5.0, 4.0)
    o.fill_(float("nan"))
    _call("mvr_transform_blending", 0, _box(img.shape), bo, bl, _aff(), BB, _box(out), _p(o))
    assert np.array_equal(o.cpu().numpy(),
                          hip.transform_blending(img.shape, tuple(bo), tuple(bl), AFFINE, tuple(BB), out))


@pytest.mark.parametrize("views", [1, 4, 5])
@pytest.mark.parametrize("blend", ["none", "same", "different"])
def test_fuse_group_on_device_memory(views, blend):
    from mvr import hip
    rng = np.random.default_rng(views)
    out = (8, 21, 70)
    imgs = [rng.uniform(0, 9, (10 + j, 24, 64 + j)).astype(np.float32) for j in range(views)]
    affs = [AFFINE + 0.01 * j for j in range(views)]
    fb = None if blend == "none" else [[1.0, 1.0, 0.5, 6.0, 4.0, 3.0]] * views
    db = None if blend == "none" else fb if blend == "same" else [[0.0, 0.0, 0.0, 8.0, 8.0, 40.0]] * views
    adj = [(1.1, -0.5)] * views
    ref = hip.fuse_group(imgs, affs, tuple(BB), out, adj, fb, db)
    ts = [_dev(a) for a in imgs]
    o, w = (torch.full(out, float("nan"), device="cuda") for _ in range(2))
    f32p, f64p, i32p = (ctypes.POINTER(c) for c in (ctypes.c_float, ctypes.c_double, ctypes.c_int))

    def arr(x, dtype, ptr):
        if x is None:
            return None
        a = np.ascontiguousarray(np.asarray(x, dtype))
        keep.append(a)
        return a.ctypes.data_as(ptr)

    keep = []
    dims = [[a.shape[2], a.shape[1], a.shape[0]] for a in imgs]
    _call("mvr_fuse_group", 0, views, (ctypes.c_void_p * views)(*[t.data_ptr() for t in ts]),
          arr(dims, np.int32, i32p), arr(affs, np.float64, f64p), arr(adj, np.float64, f64p),
          arr(fb, np.float32, f32p), arr(db, np.float32, f32p), BB, _box(out), _p(o), _p(w))
    assert np.array_equal(o.cpu().numpy(), ref[0]) and np.array_equal(w.cpu().numpy(), ref[1])


def test_normalisation_and_overlapping_arrays():
    from mvr import hip
    rng = np.random.default_rng(3)
    ws = rng.uniform(0, 1.2, (3, 6, 7, 33)).astype(np.float32)
    ref = hip.normalize_weights(ws)
    t = _dev(ws)
    ptrs = (ctypes.c_void_p * 3)(*[t[v].data_ptr() for v in range(3)])
    _call("mvr_normalize_weights", 0, ptrs, 3, _box(ws.shape[1:]), 1.0, 0, 0.1, 0.05)
    assert np.array_equal(t.cpu().numpy(), ref)
    # the output of a resampling in its input's memory: read as a whole before it is written
    img = rng.uniform(0, 9, (8, 9, 30)).astype(np.float32)
    t = _dev(img)
    _call("mvr_transform_view", 0, _p(t), _box(img.shape), _aff(), BB, _box(img.shape), 1, 1.0, 0.0, 1, _p(t))
    assert np.array_equal(t.cpu().numpy(), hip.transform_view(img, AFFINE, tuple(BB), img.shape))
    torch.cuda.synchronize()
