"""Workloads of the filtering library as its users run them, for timing.

Every case is a dict of plain values.  ``prepare`` makes its seeded inputs in
HBM and the descriptors a program keeps between calls, ``run`` is one call (or
one batch) through the public entry points, ``work`` counts the bytes and
operations the call cannot do without, and ``exact`` restates the result in
64-bit torch without the library.

Most cases go through the C ABI (include/ifm.h) on device arrays, as a program
with its own arrays does; ``blur_small`` and ``default_dense`` go through the
Python package's ``imfilter``.  Axis 0 of an image is the contiguous one; its
torch tensor has the axes reversed.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "imagefiltering.jl_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import imagefiltering as IF  # noqa: E402
from imagefiltering import _lib, serving  # noqa: E402

DEV = "cuda"
BORDERS = ("replicate", "reflect", "symmetric", "circular", "fill")
ELTYPES = {"u8": IF.UInt8, "n0f8": IF.N0f8, "f32": IF.Float32, "f64": IF.Float64, "bf16": IF.BFloat16}
TORCH = {"u8": torch.uint8, "n0f8": torch.uint8, "f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16}
SIZE = {"u8": 1, "n0f8": 1, "f32": 4, "f64": 8, "bf16": 2}
FILL = 1.0  # exact in every eltype


def listed():
    return [
        # a thumbnail blurred by the drop-in imfilter: host work and launches count
        {"name": "blur_small", "kind": "blur_api", "n0": 256, "n1": 192, "dtype": "f32", "out": "f64",
         "sigma": 1.5, "border": "replicate"},
        # Gaussian smoothing of a camera frame or scan, Float32 in and out
        {"name": "blur", "kind": "blur", "n0": 4096, "n1": 3072, "dtype": "f32", "out": "f32", "sigma": 3.0,
         "border": "reflect"},
        # the benchmark's dense 15 x 15 correlation (matrix cores)
        {"name": "dense15", "kind": "dense", "n0": 4096, "n1": 4096, "dtype": "f32", "out": "f32", "k": 15,
         "border": "reflect"},
        # a small non-separable stencil on an odd-sized image, default output eltype
        {"name": "stencil5", "kind": "dense", "n0": 4001, "n1": 3001, "dtype": "f32", "out": "f64", "k": 5,
         "border": "symmetric"},
        # imfilter(img, kernel, border) with everything left to its defaults: finite scan, then FFT
        {"name": "default_dense", "kind": "dense_api", "n0": 3000, "n1": 2001, "dtype": "f32", "out": "f64", "k": 21,
         "border": "reflect"},
        # separable smoothing of a microscopy volume (the benchmark's volume)
        {"name": "volume_blur", "kind": "volume", "n0": 512, "n1": 512, "n2": 256, "dtype": "f32", "out": "f64",
         "sigma": 2.0, "border": "symmetric"},
        # recursive Gaussian of the same volume
        {"name": "volume_iir", "kind": "iir", "n0": 512, "n1": 512, "n2": 256, "dtype": "f32", "out": "f64",
         "sigma": 2.0, "border": "circular"},
        # recursive Gaussian with a wide sigma on a 4K frame (background estimation)
        {"name": "image_iir", "kind": "iir", "n0": 3840, "n1": 2160, "n2": 1, "dtype": "f32", "out": "f32",
         "sigma": 12.0, "border": "replicate"},
        # denoising of 8-bit scans by the median (the benchmark's 8192^2 image of codes)
        {"name": "median_codes", "kind": "median", "n0": 8192, "n1": 8192, "dtype": "n0f8", "k": 7,
         "border": "replicate"},
        # the same on floating-point measurements (Float64 is the language's default)
        {"name": "median_float", "kind": "median", "n0": 1537, "n1": 1025, "dtype": "f64", "k": 5,
         "border": "reflect"},
        # local minimum and maximum of 8-bit codes (morphology, local contrast)
        {"name": "extrema", "kind": "extrema", "n0": 8192, "n1": 8192, "dtype": "n0f8", "k": 9},
        # a serving batch: mixed operations on images of uneven sizes in one call
        {"name": "batch", "kind": "batch", "count": 24, "lo": 64, "hi": 2048, "mix": 20261207},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("blur_api", "blur", "dense", "dense", "dense_api", "volume", "iir", "iir", "median", "median",
                       "extrema", "batch"))
    border = rng.choice(BORDERS)
    if kind in ("blur_api", "blur"):
        hi = 320 if kind == "blur_api" else 4096
        dt = rng.choice(("f32", "f32", "bf16", "n0f8"))
        return {"kind": kind, "n0": _log(rng, 48, hi), "n1": _log(rng, 48, hi), "dtype": dt,
                "out": "bf16" if dt == "bf16" else rng.choice(("f32", "f64")), "sigma": round(rng.uniform(0.6, 8.0), 2),
                "border": border}
    if kind in ("dense", "dense_api"):
        dt = rng.choice(("f32", "f32", "bf16", "n0f8"))
        k = rng.choice((3, 5, 7, 9, 15, 17, 21, 31)) if kind == "dense" else rng.choice((7, 9, 15, 21, 31, 45))
        return {"kind": kind, "n0": _log(rng, 200, 4096), "n1": _log(rng, 200, 4096), "dtype": dt,
                "out": "f64" if kind == "dense_api" else rng.choice(("f32", "f64")), "k": k, "border": border}
    if kind == "volume":
        return {"kind": kind, "n0": _log(rng, 64, 512), "n1": _log(rng, 64, 512), "n2": _log(rng, 32, 256),
                "dtype": "f32", "out": rng.choice(("f32", "f64")), "sigma": round(rng.uniform(0.6, 3.0), 2),
                "border": border}
    if kind == "iir":
        flat = rng.random() < 0.6
        return {"kind": kind, "n0": _log(rng, 100, 4096) if flat else _log(rng, 64, 512),
                "n1": _log(rng, 100, 2304) if flat else _log(rng, 64, 512), "n2": 1 if flat else _log(rng, 32, 256),
                "dtype": rng.choice(("f32", "f32", "f64")), "out": rng.choice(("f32", "f64")),
                "sigma": round(rng.uniform(1.0, 20.0), 2), "border": border}
    if kind == "median":
        dt = rng.choice(("n0f8", "n0f8", "u8", "f32", "f64"))
        hi = {"n0f8": 8192, "u8": 8192, "f32": 4096, "f64": 1100}[dt]
        k = rng.choice((3, 5, 7, 9))
        if k == 9:
            hi = min(hi, 800)
        return {"kind": kind, "n0": _log(rng, 100, hi), "n1": _log(rng, 100, hi), "dtype": dt, "k": k,
                "border": rng.choice(BORDERS[:4])}
    if kind == "extrema":
        dt = rng.choice(("n0f8", "u8", "f32"))
        hi = 4096 if dt == "f32" else 8192
        return {"kind": kind, "n0": _log(rng, 100, hi), "n1": _log(rng, 100, hi), "dtype": dt,
                "k": rng.choice((3, 5, 7, 9, 13))}
    return {"kind": "batch", "count": rng.randint(8, 24), "lo": 64, "hi": _log(rng, 300, 2048),
            "mix": rng.randrange(1 << 30)}


# ---- arrays --------------------------------------------------------------------
def _shape(case):
    return tuple(case[k] for k in ("n0", "n1", "n2") if case.get(k, 1) != 1)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _pixels(shape, dtype, seed):
    """Pixels in [0, 1) (codes: all 256, 5% salt and pepper), axes reversed."""
    g = _gen(seed)
    size = tuple(reversed(shape))
    if dtype in ("u8", "n0f8"):
        x = torch.randint(0, 256, size, dtype=torch.uint8, device=DEV, generator=g)
        u = torch.rand(size, device=DEV, generator=g)
        return x.masked_fill_(u < 0.025, 0).masked_fill_(u > 0.975, 255)
    return torch.rand(size, device=DEV, generator=g, dtype=torch.float64 if dtype == "f64" else torch.float32).to(
        TORCH[dtype])


def _array(t, dtype):
    """ifm_array of a dense tensor (axes reversed: its last one is axis 0)."""
    a = _lib.IfmArray()
    a.ndim, a.dtype, a.device, a.data = t.dim(), ELTYPES[dtype].code, 1, t.data_ptr()
    stride = 1
    for d, n in enumerate(reversed(t.shape)):
        a.size[d], a.stride[d] = n, stride
        stride *= n
    return a


def _border(name):
    b = _lib.IfmBorder()
    b.style = {"replicate": _lib.REPLICATE, "circular": _lib.CIRCULAR, "symmetric": _lib.SYMMETRIC,
               "reflect": _lib.REFLECT, "fill": _lib.FILL}[name]
    b.fill = FILL if name == "fill" else 0.0
    return b


class _Cai:
    """A DeviceArray's memory for torch (the tensor keeps it alive)."""

    def __init__(self, a, dtype):
        self.owner = a
        typestr = {"u8": "|u1", "n0f8": "|u1", "f32": "<f4", "f64": "<f8", "bf16": "<i2"}[dtype]
        self.__cuda_array_interface__ = {"shape": tuple(reversed(a.shape)), "typestr": typestr, "version": 2,
                                         "data": (a.ptr, False), "strides": None}


def _tensor(a, dtype):
    t = torch.as_tensor(_Cai(a, dtype), device=DEV)
    return t.view(torch.bfloat16) if dtype == "bf16" else t


def _device_array(t, dtype):
    a = IF.DeviceArray(tuple(reversed(t.shape)), ELTYPES[dtype], "F")
    _tensor(a, dtype).copy_(t)
    return a


# ---- kernels ---------------------------------------------------------------------
def _dense_taps(k, seed):
    rng = np.random.default_rng(seed)
    while True:
        t = rng.standard_normal((k, k))
        if abs(t.sum()) >= 1:
            return t / t.sum()


def _sigmas(case):
    n = len(_shape(case))
    return (case["sigma"],) * 2 + ((0.75 * case["sigma"],) if n == 3 else ()) if n > 1 else (case["sigma"],)


def _factors(kern):
    keep = [np.ascontiguousarray(np.asarray(f.data.data, dtype=np.float64)) for f in kern]
    fa = (_lib.IfmFactor * len(kern))()
    for i, f in enumerate(kern):
        fa[i].axis, fa[i].len, fa[i].first = f.Npre, len(keep[i]), int(f.data.first[0])
        fa[i].taps = keep[i].ctypes.data_as(C.POINTER(C.c_double))
    return fa, keep


def _iir(kern):
    arr = (_lib.IfmIir * len(kern))()
    for i, f in enumerate(kern):
        k = f.data
        arr[i].a[:], arr[i].b[:], arr[i].M[:] = list(k.a), list(k.b), list(np.asarray(k.M).ravel())
        arr[i].scale, arr[i].axis = k.scale, f.Npre
    return arr


def _mix(case):
    return serving.request_mix(case["count"], seed=case["mix"], side=(case["lo"], case["hi"]))


def prepare(case, seed):
    kind = case["kind"]
    L, ctx = _lib.load(), _lib.ctx()
    if kind == "batch":
        mix = _mix(case)
        ins, outs, bufs = [], [], []
        for i in range(mix["n"]):
            shape = (int(mix["w"][i]), int(mix["h"][i]))
            dt = "bf16" if mix["dtype"][i] else "f32"
            op = serving.OPS[mix["op"][i]]
            ins.append(_pixels(shape, dt, seed * 1000 + i))
            o = [torch.empty(ins[-1].shape, dtype=ins[-1].dtype if op == "median7" else torch.float64, device=DEV)
                 for _ in range(2 if op == "sobel" else 1)]
            outs.append(o)
            bufs.append((ins[-1].data_ptr(), o[0].data_ptr(), o[1].data_ptr() if len(o) > 1 else None))
        arr, keep = serving.requests(mix, bufs)
        return {"call": lambda: L.ifm_batch_run(ctx, arr, mix["n"]), "out": outs, "keep": (arr, keep, ins)}
    shape, dt = _shape(case), case["dtype"]
    img = _pixels(shape, dt, seed)
    if kind == "blur_api":
        d = _device_array(img, dt)
        kern = IF.KernelFactors.gaussian((case["sigma"],) * 2)
        border = IF.Fill(FILL) if case["border"] == "fill" else case["border"]
        T = ELTYPES[case["out"]]
        return {"api": lambda: IF.imfilter(T, d, kern, border), "dtype": case["out"]}
    if kind == "dense_api":
        d = _device_array(img, dt)
        kern = IF.centered(_dense_taps(case["k"], seed))
        border = IF.Fill(FILL) if case["border"] == "fill" else case["border"]
        return {"api": lambda: IF.imfilter(d, kern, border), "dtype": case["out"]}
    a = _array(img, dt)
    if kind == "median":
        out = torch.empty_like(img)
        ao = _array(out, dt)
        k = case["k"]
        wf, wl = _lib.i64([-(k // 2)] * 2), _lib.i64([k] * 2)
        b = _border(case["border"])
        return {"call": lambda: L.ifm_mapwindow_median(ctx, a, ao, None, wf, wl, b), "out": out, "keep": img}
    if kind == "extrema":
        out = [torch.empty_like(img), torch.empty_like(img)]
        a0, a1 = _array(out[0], dt), _array(out[1], dt)
        win = _lib.i64([case["k"]] * 2)
        return {"call": lambda: L.ifm_extrema_filter(ctx, a, a0, a1, win), "out": out, "keep": img}
    out = torch.empty(img.shape, dtype=TORCH[case["out"]], device=DEV)
    ao = _array(out, case["out"])
    b = _border(case["border"])
    if kind == "dense":
        taps = _dense_taps(case["k"], seed)
        flat = np.ascontiguousarray(taps.ravel(order="F"))
        ks = _lib.IfmKernel()
        ks.ndim = 2
        for d in range(2):
            ks.size[d], ks.first[d] = case["k"], -(case["k"] // 2)
        ks.taps = flat.ctypes.data_as(C.POINTER(C.c_double))
        return {"call": lambda: L.ifm_imfilter_dense(ctx, a, ao, None, ks, b, _lib.PREC_AUTO), "out": out,
                "keep": (img, flat)}
    if kind == "iir":
        kern = IF.KernelFactors.IIRGaussian(_sigmas(case), False)
        ks = _iir(kern)
        return {"call": lambda: L.ifm_imfilter_iir(ctx, a, ao, ks, len(kern), b), "out": out, "keep": img}
    kern = IF.KernelFactors.gaussian(_sigmas(case))
    fa, keep = _factors(kern)
    return {"call": lambda: L.ifm_imfilter_fir(ctx, a, ao, None, fa, len(kern), b), "out": out, "keep": (img, keep)}


def run(state):
    if "api" in state:
        return _tensor(state["api"](), state["dtype"])
    _lib.check(state["call"]())
    return state["out"]


def work(case):
    kind = case["kind"]
    if kind == "batch":
        mix = _mix(case)
        px = serving.request_pixels(mix)
        taps = {"gaussian": 0, "sobel": 12, "median7": 49, "dense15": 225}
        per = [taps[serving.OPS[o]] or 2 * (4 * math.ceil(s) + 1) for o, s in zip(mix["op"], mix["sigma"])]
        return {"bytes": float(serving.request_bytes(mix).sum()), "flops": float((px * 2 * np.array(per)).sum())}
    shape = _shape(case)
    px, n = math.prod(shape), len(shape)
    ein = SIZE[case["dtype"]]
    if kind == "median":
        return {"bytes": px * 2 * ein, "flops": px * case["k"] ** 2}
    if kind == "extrema":
        return {"bytes": px * 3 * ein, "flops": px * 4 * math.ceil(math.log2(case["k"] + 1))}
    eout = SIZE[case["out"]]
    if kind in ("dense", "dense_api"):
        flops = 2 * case["k"] ** 2
        if kind == "dense_api":  # a transform of the image and one back, five operations per butterfly point
            flops = min(flops, 10 * math.log2(px))
    elif kind == "iir":
        flops = 13 * n
    else:
        s = _sigmas(case) if kind == "volume" else (case["sigma"],) * 2
        flops = sum(2 * (4 * math.ceil(v) + 1) for v in s)
    return {"bytes": px * (ein + eout), "flops": px * flops}


# ---- the same in 64 bits, by plain torch ---------------------------------------------
def _index(n, lo, hi, border):
    i = torch.arange(-lo, n + hi, device=DEV)
    if border == "replicate":
        return i.clamp(0, n - 1)
    if border == "circular":
        return i % n
    if border == "symmetric":
        j = i % (2 * n)
        return torch.where(j < n, j, 2 * n - 1 - j)
    if border == "reflect":
        j = i % max(2 * n - 2, 1)
        return torch.where(j < n, j, 2 * n - 2 - j)
    return torch.where((i >= 0) & (i < n), i, torch.full_like(i, -1))


def _extended(x, dim, h, border):
    idx = _index(x.shape[dim], h, h, border)
    y = x.index_select(dim, idx.clamp(min=0))
    if border == "fill":
        shape = [1] * x.dim()
        shape[dim] = -1
        y = torch.where((idx < 0).reshape(shape), torch.full_like(y, FILL), y)
    return y


def _gauss(sigma):
    w = 2 * math.ceil(sigma)
    x = np.arange(-w, w + 1, dtype=np.float64)
    g = np.exp(-x ** 2 / (2 * sigma ** 2))
    return g / g.sum()


def _correlate(x, taps, border):
    """The correlation with a centred 2-D kernel, taps[i, j] at axes (0, 1) = dims (1, 0)."""
    h0, h1 = taps.shape[0] // 2, taps.shape[1] // 2
    n1, n0 = x.shape
    e = _extended(_extended(x, 1, h0, border), 0, h1, border)
    out = torch.zeros_like(x)
    for j in range(taps.shape[1]):
        for i in range(taps.shape[0]):
            if taps[i, j]:
                out.add_(e[j:j + n1, i:i + n0], alpha=float(taps[i, j]))
    return out


def _correlate_axes(x, taps, border):
    """One factor per axis, every border extended from the image itself."""
    for d in range(x.dim()):
        dim = x.dim() - 1 - d
        x = _extended(x, dim, len(taps[d]) // 2, border)
    for d, t in enumerate(taps):
        dim = x.dim() - 1 - d
        n = x.shape[dim] - len(t) + 1
        y = torch.zeros_like(x.narrow(dim, 0, n))
        for i, v in enumerate(t):
            y.add_(x.narrow(dim, i, n), alpha=float(v))
        x = y
    return x


def _recursive(x, sigma, border, dim):
    """Young and van Vliet's recursive Gaussian along one axis: the signal is
    continued by its end values (or the Fill value) without end, forward from
    the steady state, then backward from the steady state."""
    m0, m1, m2 = 1.16680, 1.10783, 1.40586
    q = 1.31564 * (math.sqrt(1 + 0.490811 * sigma * sigma) - 1)
    s = (m0 + q) * (m1 * m1 + m2 * m2 + 2 * m1 * q + q * q)
    a = (q * (2 * m0 * m1 + m1 * m1 + m2 * m2 + (2 * m0 + 4 * m1) * q + 3 * q * q) / s,
         -q * q * (m0 + 2 * m1 + 3 * q) / s, q * q * q / s)
    B = (m0 * (m1 * m1 + m2 * m2) / s) ** 2
    x = x.movedim(dim, 0).contiguous()
    n, ext = x.shape[0], int(40 * sigma) + 40
    first, last = (torch.full_like(x[0], FILL),) * 2 if border == "fill" else (x[0].clone(), x[-1].clone())
    y = torch.empty((n + ext,) + tuple(x.shape[1:]), dtype=x.dtype, device=DEV)
    y1 = y2 = y3 = first / (1 - sum(a))
    for i in range(n + ext):
        t = torch.add(x[i] if i < n else last, y1, alpha=a[0], out=y[i])
        t.add_(y2, alpha=a[1]).add_(y3, alpha=a[2])
        y1, y2, y3 = t, y1, y2
    z1 = z2 = z3 = last / (1 - sum(a)) ** 2
    for i in range(n + ext - 1, -1, -1):
        t = y[i].add_(z1, alpha=a[0]).add_(z2, alpha=a[1]).add_(z3, alpha=a[2])
        z1, z2, z3 = t, z1, z2
    return (y[:n] * B).movedim(0, dim)


def _real(img, dtype):
    x = img.to(torch.float64)
    return x / 255.0 if dtype == "n0f8" else x


def exact(case, seed):
    kind = case["kind"]
    if kind == "extrema":
        return None
    if kind == "batch":
        mix = _mix(case)
        res = []
        for i in range(mix["n"]):
            shape = (int(mix["w"][i]), int(mix["h"][i]))
            img = _pixels(shape, "bf16" if mix["dtype"][i] else "f32", seed * 1000 + i)
            op = serving.OPS[mix["op"][i]]
            border = serving.BORDERS[mix["border"][i]]
            x = img.to(torch.float64)
            if border == "fill0":  # Fill(0): a ring of zeros as wide as any kernel here, cut off again
                x = torch.nn.functional.pad(x, (40, 40, 40, 40))
                border = "replicate"
            crop = slice(40, -40) if x.shape != img.shape else slice(None)
            if op == "median7":
                res.append([None])
            elif op == "gaussian":
                res.append([_correlate_axes(x, [_gauss(float(mix["sigma"][i]))] * 2, border)[crop, crop].cpu()])
            elif op == "sobel":
                d, w = np.array([-0.5, 0.0, 0.5]), np.array([0.25, 0.5, 0.25])
                res.append([_correlate_axes(x, t, border)[crop, crop].cpu() for t in ([d, w], [w, d])])
            else:
                res.append([_correlate(x, _dense_taps(15, int(mix["kseed"][i])), border)[crop, crop].cpu()])
        return res
    img = _pixels(_shape(case), case["dtype"], seed)
    if kind == "median":
        if case["dtype"] not in ("f32", "f64") or img.numel() > 6_000_000:
            return None
        k, h = case["k"], case["k"] // 2
        border = case["border"]
        if border == "circular":  # an edge window wraps inside its part of the image
            return None
        e = _extended(_extended(img, 1, h, border), 0, h, border)
        out = torch.empty_like(img)
        for r in range(0, img.shape[0], 64):
            rows = e[r:r + 64 + 2 * h]
            w = rows.unfold(0, k, 1).unfold(1, k, 1)
            out[r:r + w.shape[0]] = w.reshape(w.shape[0], w.shape[1], k * k).sort(-1).values[..., k * k // 2]
        return out.to(torch.float64)
    x = _real(img, case["dtype"])
    if kind in ("dense", "dense_api"):
        return _correlate(x, _dense_taps(case["k"], seed), case["border"])
    if kind == "iir":
        for d, s in enumerate(_sigmas(case)):
            x = _recursive(x, s, case["border"], x.dim() - 1 - d)
        return x
    s = _sigmas(case) if kind == "volume" else (case["sigma"],) * 2
    return _correlate_axes(x, [_gauss(v) for v in s], case["border"])
