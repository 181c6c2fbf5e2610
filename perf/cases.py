"""Timed cases of the framework's public entry points, from single convolutions to whole deconvolution iterations.

The kinds of case and what each stands for in use:

  conv_device  one convolution on device memory for callers that may not allocate (graph capture, serving loops)
  conv_host    one convolution of host arrays, the call that replaces the reference's native convolution
  init         the set-up of a deconvolution: second kernels, kernel spectra, initial estimate
  rl           Richardson-Lucy iterations of the resident driver (sequential, multiplicative, batched blocks)
  infer        the learned initial estimate of an initialised deconvolution
  train        one training step of the network (forward, backward, optimiser)
  prepare      input preparation: groups of views fused into the deconvolution frame, weights normalised

A case is a dict of plain values.  ``prepare`` builds what a program holds before the call from the seed, ``run`` is
one pass, ``exact`` gives the same outputs in 64 bits with torch alone, ``work`` the bytes and operations of a pass
(inputs read once, outputs written once; FFT convolutions at 5 n log2 n / 2 operations per real transform).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "multiview-reconstruction_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

from mvr import hip, learned  # noqa: E402

DEV = "cuda"
LAMBDA = 0.0006      # the reference GUI's Tikhonov parameter
MIN_VALUE = 1e-4     # MultiViewDeconvolution.minValue
NUM_THREADS = 8      # numeric thread count of the kernel normalisation
CIN = (16, 16, 16, 32, 32, 64, 96, 32, 48, 16)
COUT = (16, 16, 32, 32, 64, 64, 32, 32, 16, 16)
TAPS = [(t // 9 - 1, (t // 3) % 3 - 1, t % 3 - 1) for t in range(27)]


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: a preview-sized block in a capture or serving loop, where launches count
        dict(name="conv_device_48", kind="conv_device", nx=48, ny=40, nz=33, kx=15, ky=13, kz=11, ext="mirror"),
        # the drop-in convolution of one block of host data
        dict(name="conv_host_160", kind="conv_host", nx=160, ny=150, nz=96, kx=31, ky=31, kz=31, ext="value"),
        # set-up of a six-view Efficient-Bayesian run: compound kernels of all pairs of views, twelve spectra
        dict(name="init_eb_6views", kind="init", nx=192, ny=176, nz=128, views=6, kx=31, ky=31, kz=31,
             psf="EFFICIENT_BAYESIAN"),
        # a small crop tried out interactively: launch-bound passes
        dict(name="rl_small_64", kind="rl", nx=64, ny=60, nz=52, views=2, kx=15, ky=15, kz=21,
             psf="EFFICIENT_BAYESIAN", scheme="SEQ", iterations=5, block=0, uneven=False),
        # the benchmark's 256^3 x 6 views, Optimization-II
        dict(name="rl_256_6views", kind="rl", nx=256, ny=256, nz=256, views=6, kx=41, ky=41, kz=41,
             psf="OPTIMIZATION_II", scheme="SEQ", iterations=1, block=0, uneven=False),
        # four views of uneven extents in a common frame
        dict(name="rl_uneven_400", kind="rl", nx=400, ny=352, nz=224, views=4, kx=45, ky=45, kz=45,
             psf="EFFICIENT_BAYESIAN", scheme="SEQ", iterations=1, block=0, uneven=True),
        # a large frame with the largest PSFs in use, odd extents
        dict(name="rl_large_768", kind="rl", nx=767, ny=700, nz=321, views=2, kx=61, ky=61, kz=61,
             psf="OPTIMIZATION_I", scheme="SEQ", iterations=1, block=0, uneven=False),
        # the multiplicative scheme
        dict(name="rl_mul_160", kind="rl", nx=160, ny=150, nz=140, views=4, kx=31, ky=31, kz=31,
             psf="INDEPENDENT", scheme="MUL", iterations=2, block=0, uneven=False),
        # the reference's block structure, all blocks of a view in one launch per pass
        dict(name="rl_blocks_200", kind="rl", nx=200, ny=176, nz=112, views=4, kx=25, ky=25, kz=25,
             psf="EFFICIENT_BAYESIAN", scheme="SEQ", iterations=1, block=64, uneven=True),
        # the learned estimate at the benchmark's size, extents that are no multiple of the network's grid
        dict(name="infer_252", kind="infer", nx=254, ny=250, nz=252, views=6),
        # the training step the networks were trained with: four patches of 64^3
        dict(name="train_4x64", kind="train", patch=64, batch=4, views=6),
        # two groups of two opposing views fused into the frame
        dict(name="prepare_2x2_220", kind="prepare", nx=220, ny=200, nz=180, groups=2, per_group=2, blend=True,
             adjust=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _odd(rng, lo, hi):
    return rng.randrange(lo | 1, hi + 1, 2)


def draw(rng):
    kind = rng.choice(["conv_device", "conv_host", "init", "rl", "rl", "rl", "infer", "train", "prepare"])
    if kind in ("conv_device", "conv_host"):
        hi = 110 if kind == "conv_device" else 200
        n = [_log_int(rng, 24, hi) for _ in range(3)]
        k = [_odd(rng, 5, 31) for _ in range(3)]
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], kx=k[0], ky=k[1], kz=k[2],
                    ext=rng.choice(["mirror", "value"]))
    if kind == "init":
        k = _odd(rng, 11, 41)
        return dict(kind=kind, nx=_log_int(rng, 64, 200), ny=_log_int(rng, 64, 200), nz=_log_int(rng, 64, 160),
                    views=rng.randint(2, 6), kx=k, ky=k, kz=_odd(rng, 11, 31),
                    psf=rng.choice(["EFFICIENT_BAYESIAN", "OPTIMIZATION_I", "OPTIMIZATION_II", "INDEPENDENT"]))
    if kind == "rl":
        form = rng.choice(["seq", "seq", "seq", "mul", "blocks"])
        if form == "blocks":
            k = _odd(rng, 11, 25)
            n = [_log_int(rng, 72, 220) for _ in range(3)]
            block = rng.choice([48, 64, 80])
        else:
            n = [_log_int(rng, 48, 420 if form == "seq" else 200) for _ in range(3)]
            k = _odd(rng, 11, min(61, max(13, min(n) // 2)))
            block = 0
        big = n[0] * n[1] * n[2] > 4e6
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], views=rng.randint(2, 4 if big else 6), kx=k, ky=k,
                    kz=_odd(rng, 11, k), psf=rng.choice(["EFFICIENT_BAYESIAN", "OPTIMIZATION_I", "OPTIMIZATION_II",
                                                         "INDEPENDENT"]),
                    scheme="MUL" if form == "mul" else "SEQ", iterations=1 if big else rng.randint(1, 3), block=block,
                    uneven=rng.random() < 0.4)
    if kind == "infer":
        return dict(kind=kind, nx=_log_int(rng, 64, 256), ny=_log_int(rng, 64, 256), nz=_log_int(rng, 64, 256),
                    views=rng.choice([6, 8]))
    if kind == "train":
        patch = rng.choice([32, 40, 48, 64])
        return dict(kind=kind, patch=patch, batch=rng.randint(1, 4), views=rng.choice([3, 6, 8]))
    return dict(kind="prepare", nx=_log_int(rng, 64, 256), ny=_log_int(rng, 64, 256), nz=_log_int(rng, 64, 256),
                groups=rng.randint(2, 4), per_group=rng.randint(1, 3), blend=rng.random() < 0.7,
                adjust=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs
def _generator(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1009 + salt)
    return g


def _phantom(shape, g):
    """A few bright smooth structures on a background of 10, in photons."""
    coarse = [max(2, s // 6) for s in shape]
    f = torch.rand(coarse, generator=g, device=DEV) ** 8 * 500.0
    f = torch.nn.functional.interpolate(f[None, None], size=tuple(shape), mode="trilinear", align_corners=True)[0, 0]
    return (f + 10.0).contiguous()


def _views(shape, V, seed, uneven=False):
    """V noisy views of one phantom, each blurred along one axis, and their normalised blending weights (cosine ramps
    at the z faces); uneven: each view covers a centred box of its own, image and weight 0 outside."""
    g = _generator(seed)
    ph = _phantom(shape, g)
    imgs, ws = [], []
    for v in range(V):
        k = [1, 1, 1]
        k[v % 3] = 5
        b = torch.nn.functional.avg_pool3d(ph[None, None], k, stride=1, padding=[a // 2 for a in k],
                                           count_include_pad=False)[0, 0]
        img = torch.poisson(b, generator=g)
        nz = shape[0]
        z = torch.arange(nz, device=DEV, dtype=torch.float32)
        d = torch.minimum(z + 1 + v % 3, nz - z) / max(4.0, min(20.0, nz / 4.0))
        w = (0.5 - 0.5 * torch.cos(math.pi * d.clamp(0, 1)))[:, None, None].expand(*shape).contiguous()
        if uneven:
            mask = torch.zeros(shape, device=DEV)
            cut = [int(s * 0.04 * ((v + a) % 3)) for a, s in enumerate(shape)]
            mask[cut[0]:shape[0] - cut[0], cut[1]:shape[1] - cut[1], cut[2]:shape[2] - cut[2]] = 1.0
            img = img * mask
            w = w * mask
        imgs.append(img.contiguous())
        ws.append(w)
    total = sum(ws).clamp(min=1.0)
    return imgs, [(w / total).contiguous() for w in ws]


def _psfs(kshape, V, seed):
    """Anisotropic Gaussians rotated about y, one per view (float32, [z, y, x])."""
    r = np.random.default_rng(seed)
    out = []
    for v in range(V):
        t = math.pi * (v + 0.2 * r.random()) / V
        sxy, sz = max(0.8, min(kshape) / 22.0) * (1 + 0.1 * r.random()), max(1.2, min(kshape) / 8.0)
        rot = np.array([[math.cos(t), 0, math.sin(t)], [0, 1, 0], [-math.sin(t), 0, math.cos(t)]])
        icov = np.linalg.inv(rot @ np.diag([sxy ** 2, sxy ** 2, sz ** 2]) @ rot.T)
        z, y, x = np.meshgrid(*[np.arange(k) - k // 2 for k in kshape], indexing="ij")
        p = np.stack([x, y, z], -1).astype(np.float64)
        k = np.exp(-0.5 * ((p @ icov) * p).sum(-1))
        out.append((k / k.sum()).astype(np.float32))
    return out


def _shape(c):
    return (c["nz"], c["ny"], c["nx"])


def _kshape(c):
    return (c["kz"], c["ky"], c["kx"])


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _conv_inputs(case, seed):
    g = _generator(seed)
    img = torch.poisson(_phantom(_shape(case), g), generator=g)
    return img, _psfs(_kshape(case), 1, seed)[0]


def _deconvolution(case, seed, init=True):
    shape = _shape(case)
    imgs, ws = _views(shape, case["views"], seed, case.get("uneven", False))
    d = hip.Decon(shape, case["views"], case.get("psf", "OPTIMIZATION_II"), case.get("scheme", "SEQ"), LAMBDA,
                  MIN_VALUE, NUM_THREADS)
    psfs = _psfs(_kshape(case), case["views"], seed)
    torch.cuda.synchronize()
    for v in range(case["views"]):
        d.set_view_device(v, imgs[v].data_ptr(), ws[v].data_ptr(), psfs[v])
    if case.get("block"):
        d.set_block_size([case["block"] + 2 * (case[k] - 1) for k in ("kx", "ky", "kz")])
    if init:
        d.init()
    return dict(d=d, psi=torch.empty(shape, device=DEV))


def _psi(s):
    """The handle's psi, in device memory of the caller's."""
    if hip.lib().mvr_decon_get_psi(s["d"].h, _ptr(s["psi"])) < 0:
        raise RuntimeError(hip.lib().mvr_last_error().decode())
    return s["psi"]


def _network_case(case):
    return dict(case, kx=5, ky=5, kz=5)


def _weights_file(case):
    return learned.DEFAULT_WEIGHTS if case["views"] == 6 else learned.TRAINING["c5"][1]


def _train_inputs(case, seed):
    p = case["patch"]
    shape = (p + 9, p + 14, p + 11)
    vols = []
    for i in range(2):
        imgs, ws = _views(shape, case["views"], 2 * seed + i)
        target = _phantom(shape, _generator(2 * seed + i))
        vols.append(([a.cpu().numpy() for a in imgs], [a.cpu().numpy() for a in ws], target.cpu().numpy()))
    r = np.random.default_rng(seed)
    origins = [[int(r.integers(0, s - p + 1)) for s in shape] for _ in range(case["batch"])]
    return vols, [b % 2 for b in range(case["batch"])], origins


def _network_start(case, seed):
    """He-normal weights of a network before its training, small biases (one flat vector in layer order)."""
    r = np.random.default_rng(seed + 17)
    parts = []
    for l in range(10):
        w = r.normal(0, math.sqrt(2.0 / (27 * (case["views"] + 1 if l == 0 else CIN[l]))), (27, COUT[l], CIN[l]))
        if l == 0:
            w[:, :, case["views"] + 1:] = 0
        parts += [w.ravel(), r.normal(0, 0.05, COUT[l])]
    parts.append(np.append(r.normal(0, 0.1, 16), 0.01))
    return np.concatenate(parts).astype(np.float32)


def _group_inputs(case, seed):
    """Groups of opposing views: images a little smaller than the frame, registrations (small rotation about y, scale,
    shift), intensity adjustments, blending borders and ranges."""
    shape = _shape(case)
    box = (case["nx"], case["ny"], case["nz"])
    r = np.random.default_rng(seed)
    groups = []
    for i in range(case["groups"]):
        views = []
        for j in range(case["per_group"]):
            n = [max(8, int(s * r.uniform(0.8, 0.95))) for s in shape]
            g = _generator(seed, 100 * i + j)
            img = torch.poisson(_phantom(n, g), generator=g)
            t = math.radians(r.uniform(-8, 8) + 90.0 * i)
            rot = np.array([[math.cos(t), 0, math.sin(t)], [0, 1, 0], [-math.sin(t), 0, math.cos(t)]])
            a = rot @ np.diag(r.uniform(0.97, 1.05, 3))
            centre = np.array([n[2], n[1], n[0]]) / 2.0
            shift = np.array(box) / 2.0 + r.uniform(-4, 4, 3) - a @ centre
            views.append(dict(img=img, affine=np.concatenate([a, shift[:, None]], 1),
                              adjust=(r.uniform(0.9, 1.1), r.uniform(-2, 2))))
        groups.append(views)
    return groups, np.array([2.5, 2.0, 3.0], np.float32), np.array([14.0, 12.0, 16.0], np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "conv_device":
        img, k = _conv_inputs(case, seed)
        return dict(kind=kind, ext=case["ext"], img=img, k=torch.from_numpy(k).to(DEV), out=torch.empty_like(img))
    if kind == "conv_host":
        img, k = _conv_inputs(case, seed)
        return dict(kind=kind, ext=case["ext"], img=img.cpu().numpy(), k=k)
    if kind == "init":
        return dict(_deconvolution(case, seed, init=False), kind=kind, V=case["views"], kshape=_kshape(case))
    if kind == "rl":
        return dict(_deconvolution(case, seed), kind=kind, iterations=case["iterations"])
    if kind == "infer":
        s = _deconvolution(_network_case(case), seed)
        return dict(s, kind=kind, net=learned.load(_weights_file(case)))
    if kind == "train":
        vols, index, origins = _train_inputs(case, seed)
        net = hip.UNet(case["views"], seed=seed)
        net.set_params(_network_start(case, seed))
        for v in vols:
            net.add_volume(*v)
        return dict(kind=kind, net=net, index=index, origins=origins, patch=case["patch"])
    groups, border, ramp = _group_inputs(case, seed)
    shape = _shape(case)
    calls = []
    for views in groups:
        n = len(views)
        calls.append(dict(
            keep=views, n=n, imgs=(ctypes.c_void_p * n)(*[v["img"].data_ptr() for v in views]),
            dims=np.array([v["img"].shape[::-1] for v in views], np.int32),
            affines=np.array([v["affine"] for v in views], np.float64).reshape(n, 12),
            adjust=np.array([v["adjust"] for v in views], np.float64) if case["adjust"] else None,
            blend=np.tile(np.concatenate([border, ramp]), (n, 1)).astype(np.float32) if case["blend"] else None))
    G = len(groups)
    return dict(kind=kind, calls=calls, G=G, imgs=torch.empty((G,) + shape, device=DEV),
                ws=torch.empty((G,) + shape, device=DEV), shape=shape)


# ------------------------------------------------------------------ one pass
def _check(rc):
    if rc < 0:
        raise RuntimeError(hip.lib().mvr_last_error().decode())


def run(state):
    s = state
    kind = s["kind"]
    if kind == "conv_device":
        hip.fft_convolve_noalloc(s["img"].data_ptr(), tuple(s["img"].shape), s["k"].data_ptr(), tuple(s["k"].shape),
                                 s["out"].data_ptr(), ext=s["ext"], value=1.0)
        return s["out"]
    if kind == "conv_host":
        return hip.fft_convolve(s["img"], s["k"], ext=s["ext"], value=1.0)
    if kind == "init":
        s["d"].init()
        ks = [s["d"].kernels(v, s["kshape"]) for v in range(s["V"])]
        return dict(psi=_psi(s), k1=[k[0] for k in ks], k2=[k[1] for k in ks])
    if kind == "rl":
        s["d"].reset_psi()
        s["d"].run(s["iterations"])
        return _psi(s)
    if kind == "infer":
        s["d"].init_learned(s["net"])
        return _psi(s)
    if kind == "train":
        # learning rate 0, the first step of a warm-up: the optimiser runs and a pass can be repeated
        loss = s["net"].train_step(s["index"], s["origins"], s["patch"], 0.0)
        return dict(loss=np.float32(loss), grads=s["net"].grads())
    lib = hip.lib()
    f32p, f64p, i32p = (ctypes.POINTER(t) for t in (ctypes.c_float, ctypes.c_double, ctypes.c_int))
    bb = (ctypes.c_longlong * 3)(0, 0, 0)
    nz, ny, nx = s["shape"]
    dims = (ctypes.c_int * 3)(nx, ny, nz)
    for g, c in enumerate(s["calls"]):
        adjust = None if c["adjust"] is None else c["adjust"].ctypes.data_as(f64p)
        blend = None if c["blend"] is None else c["blend"].ctypes.data_as(f32p)
        _check(lib.mvr_fuse_group(0, c["n"], c["imgs"], c["dims"].ctypes.data_as(i32p),
                                  c["affines"].ctypes.data_as(f64p), adjust, blend, blend, bb, dims,
                                  _ptr(s["imgs"][g]), _ptr(s["ws"][g])))
    ptrs = (ctypes.c_void_p * s["G"])(*[s["ws"][g].data_ptr() for g in range(s["G"])])
    _check(lib.mvr_normalize_weights(0, ptrs, s["G"], dims, 1.0, 0, 0.1, 0.05))
    return dict(imgs=s["imgs"], weights=s["ws"])


# ------------------------------------------------------------------ bytes and operations of a pass
def _conv_flops(n, k):
    e = 1.0
    for a, b in zip(n, k):
        e *= a + b - 1
    return 2 * 2.5 * e * math.log2(e) + 3 * e     # forward and inverse real transform, spectrum product


def _network_flops(vox, V):
    level = (1, 1, 8, 8, 64, 64, 8, 8, 1, 1)
    return sum(2.0 * 27 * (V + 1 if l == 0 else CIN[l]) * COUT[l] * vox / level[l] for l in range(10))


def work(case):
    kind = case["kind"]
    if kind == "train":
        vox = case["batch"] * case["patch"] ** 3
        params = sum(27 * a * b + b for a, b in zip(CIN, COUT)) + 17
        return dict(bytes=4.0 * (vox * (2 * case["views"] + 1) + 8 * params), flops=3 * _network_flops(vox, case["views"]))
    n, vox = _shape(case), float(np.prod(_shape(case)))
    if kind in ("conv_device", "conv_host"):
        return dict(bytes=4.0 * (2 * vox + np.prod(_kshape(case))), flops=_conv_flops(n, _kshape(case)) * 1.5)
    if kind == "infer":
        return dict(bytes=4.0 * vox * (2 * case["views"] + 2), flops=_network_flops(vox, case["views"]))
    if kind == "prepare":
        views = case["groups"] * case["per_group"]
        return dict(bytes=4.0 * vox * (0.7 * views + 2 * case["groups"]), flops=vox * views * 60.0)
    V, nk = case["views"], float(np.prod(_kshape(case)))
    if kind == "init":
        pairs = {"EFFICIENT_BAYESIAN": 2 * V * (V - 1), "OPTIMIZATION_I": V * (V - 1)}.get(case["psf"], 0)
        spectra = 2 * V * 2.5 * vox * math.log2(vox)
        return dict(bytes=4.0 * (vox * (V + 1) + 4 * V * nk) + 2 * V * 4.0 * vox,
                    flops=pairs * 1.5 * _conv_flops(_kshape(case), _kshape(case)) + spectra)
    updates = case["iterations"] * V
    return dict(bytes=4.0 * (vox * (2 + 2 * V) + 2 * V * nk), flops=updates * (2 * _conv_flops(n, _kshape(case)) + 30 * vox))


# ------------------------------------------------------------------ the same in 64 bits
def _fft_length(n):
    while True:
        m = n
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n += 1


def _mirror(n, lo, hi):
    p = torch.arange(-lo, n + hi, device=DEV)
    if n == 1:
        return torch.zeros_like(p)
    p = p.remainder(2 * n - 2)
    return torch.where(p >= n, 2 * n - 2 - p, p)


def _extend(a, kshape, ext, value):
    lo = [k - 1 - k // 2 for k in kshape]
    hi = [k // 2 for k in kshape]
    if ext == "mirror":
        for d in range(3):
            a = a.index_select(d, _mirror(a.shape[d], lo[d], hi[d]))
        return a
    out = torch.full([n + l + h for n, l, h in zip(a.shape, lo, hi)], float(value), device=DEV, dtype=torch.float64)
    out[lo[0]:lo[0] + a.shape[0], lo[1]:lo[1] + a.shape[1], lo[2]:lo[2] + a.shape[2]] = a
    return out


def _spectrum(k, n):
    length = [_fft_length(a + b - 1) for a, b in zip(n, k.shape)]
    return torch.fft.rfftn(k.double().to(DEV), s=length), length, tuple(k.shape)


def _convolve(a, spec, ext, value=0.0):
    """out[p] = sum_j k[j] ext(a)[p + K / 2 - j], kernel centre K / 2."""
    f, length, ks = spec
    n = a.shape
    e = torch.fft.rfftn(_extend(a, ks, ext, value), s=length)
    e *= f
    r = torch.fft.irfftn(e, s=length)
    return r[ks[0] - 1:ks[0] - 1 + n[0], ks[1] - 1:ks[1] - 1 + n[1], ks[2] - 1:ks[2] - 1 + n[2]].contiguous()


def _norm_sum(k):
    """The kernel over its sum, to which the reference adds the first portion's sum once more."""
    flat = k.reshape(-1)
    n = flat.numel()
    parts = n if n <= NUM_THREADS else max(NUM_THREADS, n // 64 ** 3)
    return k / (flat.sum() + flat[:n // parts].sum())


def _kernels(psfs, kind):
    flip = lambda a: torch.flip(a, (0, 1, 2))  # noqa: E731  (odd sizes)
    k1 = [_norm_sum(torch.from_numpy(k).to(DEV).double()) for k in psfs]
    V, k2 = len(k1), []
    same = lambda a, b: _convolve(a, _spectrum(b, a.shape), "value", 0.0)  # noqa: E731
    for v in range(V):
        if V == 1 or kind == "INDEPENDENT":
            k2.append(flip(k1[v]))
        elif kind == "EFFICIENT_BAYESIAN":
            t = flip(k1[v])
            for w in range(V):
                if w != v:
                    t = t * same(same(flip(k1[v]), k1[w]), flip(k1[w]))
            k2.append(_norm_sum(t))
        elif kind == "OPTIMIZATION_I":
            t = k1[v]
            for w in range(V):
                if w != v:
                    t = t * same(k1[v], flip(k1[w]))
            k2.append(flip(_norm_sum(t)))
        else:
            k2.append(flip(_norm_sum(k1[v] ** V)))
    return k1, k2


def _average(imgs):
    total, count = torch.zeros_like(imgs[0], dtype=torch.float64), torch.zeros_like(imgs[0], dtype=torch.float64)
    for a in imgs:
        total += torch.where(a > 0, a.double(), 0.0)
        count += (a > 0).double()
    some = count > 0
    return float((total[some] / count[some]).sum() / some.sum())


def _next(value, mx, lam):
    lo = float(np.float32(MIN_VALUE))
    t = (torch.sqrt(1.0 + 2.0 * lam * value.clamp(min=0) / mx) - 1.0) / lam * mx
    return torch.where(value > 0, t, lo).clamp(min=lo)


def _exact_rl(case, seed):
    imgs, ws = _views(_shape(case), case["views"], seed, case["uneven"])
    k1, k2 = _kernels(_psfs(_kshape(case), case["views"], seed), case["psf"])
    n = _shape(case)
    lam = float(np.float32(LAMBDA))
    psi = torch.full(n, _average(imgs), device=DEV, dtype=torch.float64)
    tops = [float(a.max()) for a in imgs]
    s1 = [_spectrum(k, n) for k in k1]
    s2 = [_spectrum(k, n) for k in k2]
    for _ in range(case["iterations"]):
        product = None
        for v in range(case["views"]):
            blurred = _convolve(psi, s1[v], "mirror")
            img = imgs[v].double()
            back = _convolve(torch.where(img > 0, img / blurred, 1.0), s2[v], "value", 1.0)
            if case["scheme"] == "SEQ":
                psi = psi + (_next(psi * back, tops[v], lam) - psi) * ws[v].double()
            else:
                product = back if product is None else product * back
        if case["scheme"] == "MUL":
            total = sum(w.double() for w in ws).clamp(max=1.0)
            mean = product ** (1.0 / case["views"])
            psi = psi + (_next(psi * mean, float(np.float32(np.mean(tops))), lam) - psi) * total
    return psi


def _conv3(x, w):
    """[N, D, H, W, Ci] with [27, Co, Ci], zero padding."""
    n, d, h, wd, _ = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = None
    for t, (dz, dy, dx) in enumerate(TAPS):
        p = xp[:, 1 + dz:1 + dz + d, 1 + dy:1 + dy + h, 1 + dx:1 + dx + wd] @ w[t].T
        out = p if out is None else out.add_(p)
    return out


class _Conv3(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        return _conv3(x, w)

    @staticmethod
    def backward(ctx, gout):
        x, w = ctx.saved_tensors
        n, d, h, wd, ci = x.shape
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        g2 = gout.reshape(-1, gout.shape[-1])
        gw = torch.stack([g2.T @ xp[:, 1 + dz:1 + dz + d, 1 + dy:1 + dy + h, 1 + dx:1 + dx + wd].reshape(-1, ci)
                          for dz, dy, dx in TAPS])
        return _conv3(gout.contiguous(), torch.flip(w, (0,)).transpose(1, 2)), gw


def _network(x0, avg, params):
    """The U-Net in 64 bits; params: list of (w, b) for the ten layers and the head."""
    conv = lambda x, l: torch.relu(_Conv3.apply(x, params[l][0]) + params[l][1])  # noqa: E731

    def pool(x):
        n, d, h, w, c = x.shape
        return x.reshape(n, d // 2, 2, h // 2, 2, w // 2, 2, c).mean(dim=(2, 4, 6))

    def up(x):
        return x.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)

    e1 = conv(conv(x0, 0), 1)
    e2 = conv(conv(pool(e1), 2), 3)
    b3 = conv(conv(pool(e2), 4), 5)
    d2 = conv(conv(torch.cat([up(b3), e2], -1), 6), 7)
    d1 = conv(conv(torch.cat([up(d2), e1], -1), 8), 9)
    wo, bo = params[10]
    return avg + d1 @ wo + bo


def _unpack(flat):
    flat = torch.from_numpy(np.asarray(flat, np.float32)).to(DEV).double()
    out, at = [], 0
    for a, b in zip(CIN, COUT):
        n = 27 * a * b
        out.append((flat[at:at + n].reshape(27, b, a), flat[at + n:at + n + b]))
        at += n + b
    return out + [(flat[at:at + 16], flat[at + 16])]


def _network_input(imgs, ws, scale):
    x = torch.zeros(tuple(imgs[0].shape) + (16,), device=DEV, dtype=torch.float64)
    s, sw = 0.0, 0.0
    for v, (a, w) in enumerate(zip(imgs, ws)):
        x[..., v] = a.double() * w.double() / scale
        s = s + x[..., v]
        sw = sw + w.double()
    avg = torch.where(sw > 0, s / sw, 0.0)
    x[..., len(imgs)] = avg
    return x, avg


def _mean_intensity(imgs, ws):
    a = sum(float((i.double() * w.double()).sum()) for i, w in zip(imgs, ws))
    b = sum(float(w.double().sum()) for w in ws)
    return max(1e-6, a / b if b > 0 else 1.0)


def _exact_infer(case, seed):
    imgs, ws = _views(_shape(case), case["views"], seed)
    scale = _mean_intensity(imgs, ws)
    full = [-(-s // 4) * 4 for s in _shape(case)]
    for d in range(3):   # positions past the last voxel repeat it
        at = torch.arange(full[d], device=DEV).clamp(max=_shape(case)[d] - 1)
        imgs = [a.index_select(d, at) for a in imgs]
        ws = [a.index_select(d, at) for a in ws]
    x, avg = _network_input(imgs, ws, scale)
    with torch.no_grad():
        pred = _network(x[None], avg[None], _unpack(np.load(_weights_file(case), allow_pickle=False)["params"]))[0]
    nz, ny, nx = _shape(case)
    return (scale * pred).clamp(min=float(np.float32(MIN_VALUE)))[:nz, :ny, :nx].contiguous()


def _exact_train(case, seed):
    vols, index, origins = _train_inputs(case, seed)
    p = case["patch"]
    xs, avgs, targets = [], [], []
    for b, (z, y, x) in zip(index, origins):
        imgs, ws, target = ([torch.from_numpy(a).to(DEV) for a in vols[b][0]],
                            [torch.from_numpy(a).to(DEV) for a in vols[b][1]], torch.from_numpy(vols[b][2]).to(DEV))
        scale = _mean_intensity(imgs, ws)
        cut = lambda a: a[z:z + p, y:y + p, x:x + p]  # noqa: E731
        x0, avg = _network_input([cut(a) for a in imgs], [cut(a) for a in ws], scale)
        xs.append(x0)
        avgs.append(avg)
        targets.append(cut(target).double() / scale)
    params = [tuple(t.requires_grad_() for t in pair) for pair in _unpack(_network_start(case, seed))]
    loss = (_network(torch.stack(xs), torch.stack(avgs), params) - torch.stack(targets)).square().mean()
    grads = torch.autograd.grad(loss, [t for pair in params for t in pair])
    return dict(loss=loss.detach(), grads=torch.cat([g.reshape(-1) for g in grads]))


def _blend_table():
    d = 0.0
    lut = np.zeros(1001)
    while d <= 1.0001:
        lut[int(d * 1000.0 + 0.5)] = (math.cos((1 - d) * math.pi) + 1) / 2
        d += 0.001
    return torch.from_numpy(lut).to(DEV)


def _exact_prepare(case, seed):
    groups, border, ramp = _group_inputs(case, seed)
    lut = _blend_table()
    grid = [torch.arange(s, device=DEV, dtype=torch.float64) for s in _shape(case)]
    out, weights = [], []
    for views in groups:
        si = sw = sd = 0.0
        for v in views:
            inv = np.linalg.inv(v["affine"][:, :3])
            off = -inv @ v["affine"][:, 3]
            t = [inv[r, 0] * grid[2][None, None, :] + inv[r, 1] * grid[1][None, :, None]
                 + inv[r, 2] * grid[0][:, None, None] + off[r] for r in range(3)]
            n = v["img"].shape[::-1]
            if case["blend"]:
                w = torch.ones_like(t[0])
                zero = torch.zeros_like(t[0], dtype=torch.bool)
                for d in range(3):
                    dist = torch.minimum(t[d] - float(border[d]), n[d] - 1 - t[d] - float(border[d]))
                    rel = dist / float(ramp[d])
                    w = torch.where(rel < 1, w * lut[(rel.clamp(0, 1) * 1000.0 + 0.5).long()], w)
                    zero |= dist <= 0
                w = torch.where(zero, 0.0, w)
            else:
                w = torch.ones_like(t[0])
            img = v["img"].double()
            if case["adjust"]:
                img = img * v["adjust"][0] + v["adjust"][1]
            inside = torch.ones_like(t[0], dtype=torch.bool)
            for d in range(3):
                inside &= (t[d] > 0) & (t[d] < n[d] - 1)
            c = [x.floor().long().clamp(0, m - 2) for x, m in zip(t, n)]
            f = [x - i for x, i in zip(t, c)]
            val = 0.0
            for dz in (0, 1):
                for dy in (0, 1):
                    for dx in (0, 1):
                        part = img[c[2] + dz, c[1] + dy, c[0] + dx]
                        for q, e in zip(f, (dx, dy, dz)):
                            part = part * (q if e else 1 - q)
                        val = val + part
            val = torch.where(inside, val.clamp(min=1.0), 0.0)
            si, sw, sd = si + val * w, sw + w, sd + w
        out.append(torch.where(sw > 0, si / sw, 0.0))
        weights.append(sd)
    w = torch.stack(weights).clamp(max=1.0)
    return dict(imgs=torch.stack(out), weights=w / w.sum(0).clamp(min=1.0))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("conv_device", "conv_host"):
        img, k = _conv_inputs(case, seed)
        return _convolve(img.double(), _spectrum(torch.from_numpy(k), img.shape), case["ext"], 1.0)
    if kind == "init":
        imgs, _ = _views(_shape(case), case["views"], seed)
        k1, k2 = _kernels(_psfs(_kshape(case), case["views"], seed), case["psf"])
        return dict(psi=torch.full(_shape(case), _average(imgs), device=DEV, dtype=torch.float64), k1=k1, k2=k2)
    return {"rl": _exact_rl, "infer": _exact_infer, "train": _exact_train, "prepare": _exact_prepare}[kind](case, seed)
