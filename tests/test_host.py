"""CPU tests of the host layer (no GPU): kernel constructors, border types,
eltype rules, dispatch decisions, and that libifm loads and exports every
entry point declared in include/ifm.h."""
import ctypes
import os
import re

import numpy as np
import pytest

import imagefiltering as IF
from imagefiltering import Kernel, KernelFactors, _lib
from imagefiltering.border import _range
from imagefiltering.eltypes import Float32, Float64, N0f8, UInt8, mul_type

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# ---- C ABI -----------------------------------------------------------------------------
def test_libifm_exports_every_declared_symbol():
    hdr = open(os.path.join(REPO, "include", "ifm.h")).read()
    declared = set(re.findall(r"\b(ifm_[a-z0-9_]+)\s*\(", hdr))
    assert len(declared) >= 20
    lib = ctypes.CDLL(_lib.LIBPATH)
    missing = [s for s in sorted(declared) if not hasattr(lib, s)]
    assert not missing, missing
    assert set(_lib.EXPORTS) <= declared


def test_libifm_version_and_device_count_without_gpu():
    L = _lib.load()
    assert L.ifm_version().startswith(b"ifm ")
    n = ctypes.c_int(-1)
    assert L.ifm_device_count(ctypes.byref(n)) == 0
    assert n.value >= 0


def test_struct_layouts_match_header():
    assert ctypes.sizeof(_lib.IfmArray) == 88
    assert ctypes.sizeof(_lib.IfmBorder) == 80
    assert ctypes.sizeof(_lib.IfmFactor) == 24
    assert ctypes.sizeof(_lib.IfmKernel) == 80
    assert ctypes.sizeof(_lib.IfmIir) == 16 * 8 + 8


# ---- kernel factories ------------------------------------------------------------------
def gaussiancmp(sigma, xr):
    c = np.exp(-np.asarray(xr, dtype=float) ** 2 / (2 * sigma ** 2))
    return c / c.sum()


def test_gaussian_factors_specialty_jl():
    k = KernelFactors.gaussian(2, 9)
    assert k.first == (-4,)
    np.testing.assert_allclose(k.data, gaussiancmp(2, range(-4, 5)), rtol=1e-14)
    kk = KernelFactors.gaussian((2, 3), (9, 7))
    np.testing.assert_allclose(kk[0].data.data, gaussiancmp(2, range(-4, 5)), rtol=1e-14)
    np.testing.assert_allclose(kk[1].data.data, gaussiancmp(3, range(-3, 4)), rtol=1e-14)
    assert abs(KernelFactors.gaussian(5).data.sum() - 1) < 1e-14
    g3 = KernelFactors.gaussian((3.0, 3.0))
    assert [len(f) for f in g3] == [13, 13] and g3[0].Npre == 0 and g3[1].Npre == 1
    k = KernelFactors.gaussian((3, 3, 0))
    assert k[2].data.data.tolist() == [1.0] and k[2].data.first == (0,)


def test_kernel_gaussian_and_dog_log():
    k = Kernel.gaussian((2, 3), (9, 7))
    np.testing.assert_allclose(k.data, np.outer(gaussiancmp(2, range(-4, 5)), gaussiancmp(3, range(-3, 4))),
                               rtol=1e-14)
    assert abs(Kernel.gaussian(5).data.sum() - 1) < 1e-12
    d = Kernel.DoG((2, 3), (4, 3.5), (9, 7))
    k1 = np.outer(gaussiancmp(2, range(-4, 5)), gaussiancmp(3, range(-3, 4)))
    k2 = np.outer(gaussiancmp(4, range(-4, 5)), gaussiancmp(3.5, range(-3, 4)))
    np.testing.assert_allclose(d.data, k1 - k2, atol=1e-15)
    assert abs(Kernel.DoG(5).data.sum()) < 1e-8
    L = Kernel.LoG(2.0)
    assert L.shape == (17, 17) and L.first == (-8, -8)
    # the LoG closed form at the centre: C * (0 - 2/σ²) with C = 1/(σ² 2π)
    assert abs(L.data[8, 8] - (1 / (4 * 2 * np.pi)) * (-2 / 4)) < 1e-15
    assert L == Kernel.LoG((2.0, 2.0))


def test_sobel_kernel_equals_factor_product():
    ky, kx = Kernel.sobel()
    fy, fx = KernelFactors.sobel()
    np.testing.assert_allclose(ky.data, np.outer([-0.5, 0, 0.5], [0.25, 0.5, 0.25]))
    np.testing.assert_allclose(kx.data, np.outer([0.25, 0.5, 0.25], [-0.5, 0, 0.5]))
    assert ky.first == (-1, -1)
    np.testing.assert_allclose(fy[0].data.data, [-0.5, 0, 0.5])


def test_box_and_errors():
    assert [f.data.data.tolist() for f in KernelFactors.box(3, 5)] == [[1 / 3] * 3, [1 / 5] * 5]
    with pytest.raises(IF.ArgumentError):
        KernelFactors.box((3, 4, 5))


@pytest.mark.parametrize("sigma", [2.0, 1.5, 3.1, 10.0, 100.0])
def test_triggs_sdika_M_satisfies_eq8(sigma):
    """test/triggs.jl:19-20: M = I1 + B*M*A."""
    k = KernelFactors.IIRGaussian(sigma)
    A = np.vstack([k.a, np.eye(3)[:2]])
    B = np.vstack([k.b, np.eye(3)[:2]])
    I1 = np.zeros((3, 3))
    I1[0, 0] = 1
    np.testing.assert_allclose(k.M, I1 + B @ k.M @ A, rtol=1e-10, atol=1e-12)


def test_iirgaussian_coefficients_sigma2():
    k = KernelFactors.IIRGaussian(2.0)
    np.testing.assert_allclose(k.a, [1.07757, -0.427266, 0.0650941], rtol=1e-5)
    assert abs(k.scale - 0.0809994) < 1e-7
    k = KernelFactors.IIRGaussian(1.5)
    np.testing.assert_allclose(k.a, [0.751101, -0.211738, 0.0243229], rtol=1e-5)
    # unit DC gain: scale / ((1 - sum a)(1 - sum b)) = 1
    for s in (1.5, 2.0, 7.0):
        k = KernelFactors.IIRGaussian(s)
        assert abs(k.scale / ((1 - k.asum) * (1 - k.bsum)) - 1) < 1e-12


# ---- borders -------------------------------------------------------------------------------
def test_pad_fill_inner_constructors_border_jl():
    assert IF.Pad("replicate", [1, 2], [5, 3]) == IF.Pad("replicate", (1, 2), (5, 3))
    assert IF.Pad("circular")(np.random.rand(3, 5)) == IF.Pad("circular", (0, 0), (3, 5))
    assert IF.Pad("circular")(IF.centered(np.random.rand(3, 5))) == IF.Pad("circular", (1, 2), (1, 2))
    assert IF.Pad("symmetric")(Kernel.Laplacian()) == IF.Pad("symmetric", (1, 1), (1, 1))
    assert IF.Inner((1, 2)) == IF.Inner((1, 2), (1, 2))
    assert IF.Inner((1, 2), ()) == IF.Inner((1, 2), (0, 0))
    assert IF.Inner()(IF.centered(np.random.rand(3, 5))) == IF.Inner((1, 2), (1, 2))
    assert IF.Fill(1, (3, 2)) == IF.Fill(1, (3, 2), (3, 2))
    assert IF.Fill(-1)(IF.centered(np.random.rand(3, 5))) == IF.Fill(-1, (1, 2), (1, 2))
    assert IF.Fill(2)(Kernel.Laplacian(), np.zeros((5, 5)), IF.Algorithm.FIR()) == IF.Fill(2, (1, 1), (1, 1))


def test_borderinstance_errors():
    assert IF.borderinstance("reflect") == IF.Pad("reflect")
    with pytest.raises(IF.ArgumentError):
        IF.borderinstance("inner")
    with pytest.raises(IF.ArgumentError):
        IF.borderinstance("nonsense")


def test_padfft_lengths():
    img = np.zeros((4096, 4096))
    p = IF.Pad("reflect")(IF.centered(np.zeros((15, 15))), img, IF.Algorithm.FFT())
    assert p.lo == (7, 7) and 7 + 4096 + p.hi[0] == 4374


@pytest.mark.parametrize("style", ["replicate", "circular", "symmetric", "reflect"])
def test_padindex_host_matches_numpy(style):
    mode = {"replicate": "edge", "circular": "wrap", "symmetric": "symmetric", "reflect": "reflect"}[style]
    for n in range(2, 7):
        for lo, hi in [(0, 0), (3, 1), (9, 13)]:
            np.testing.assert_array_equal(IF.padindex(IF.Pad(style), lo, n, hi),
                                          np.pad(np.arange(n), (lo, hi), mode=mode))


@pytest.mark.parametrize("style", ["replicate", "circular", "symmetric", "reflect"])
def test_borderarray_lazy_getindex_single_reflection(style):
    from oracle import oracle as O
    A = np.random.default_rng(1).standard_normal((5, 5))
    B = IF.BorderArray(A, IF.Pad(style, (2, 3), (4, 1)))
    P = O.padarray(A, style, [2, 3], [4, 1])    # pad < n: one reflection == periodic table
    for i in range(-2, 9):
        for j in range(-3, 6):
            assert B[i, j] == P[i + 2, j + 3]


def test_borderarray_fill_convert_errors():
    with pytest.raises(IF.ArgumentError):
        IF.BorderArray(np.zeros(3), IF.Fill(0.0))          # Fill{0}: no padding sizes
    with pytest.raises(IF.ArgumentError):
        IF.BorderArray(np.zeros(3), IF.Fill(None, (1,)))   # nothing does not convert
    with pytest.raises(IF.ArgumentError):
        IF.BorderArray(np.zeros(3, dtype=np.uint8), IF.Fill(7.5, (1,)))


# ---- eltype rules and dispatch -----------------------------------------------------------------
def test_filter_type_rules():
    assert IF.filter_type(Float32, KernelFactors.gaussian((3.0, 3.0))) is Float64
    assert IF.filter_type(Float32, (IF.centered(np.ones(3, np.float32)),)) is Float32
    assert IF.filter_type(UInt8, (IF.centered(np.ones(3)),)) is Float64
    assert IF.filter_type(N0f8, (IF.centered(np.ones(3, np.float32)),)) is Float32
    assert mul_type(N0f8, Float64) is Float64
    assert IF.filter_type(Float32, (Kernel.Laplacian(),)) is Float32


def test_factorkernel_svd():
    k = IF.factorkernel(IF.centered(np.outer([1.0, 2, 1], [-1.0, 0, 1])))
    assert len(k) == 2 and k[0].shape == (3, 1) and k[1].shape == (1, 3)
    np.testing.assert_allclose(np.outer(k[0].data.ravel(), k[1].data.ravel()), np.outer([1.0, 2, 1], [-1.0, 0, 1]),
                               atol=1e-12)
    rng = np.random.default_rng(0)
    k = IF.factorkernel(IF.centered(rng.standard_normal((15, 15))))
    assert len(k) == 1 and k[0].shape == (15, 15)
    assert len(IF.factorkernel(Kernel.LoG(2.0))) == 1


def test_filter_algorithm_heuristic():
    v = np.random.rand(100)
    k31 = (IF.centered(np.ones(31)),)
    assert IF.filter_algorithm(v, k31) == IF.Algorithm.FFT()
    w = v.copy()
    w[5] = np.nan
    assert IF.filter_algorithm(w, k31) == IF.Algorithm.FIR()
    assert IF.filter_algorithm(v, KernelFactors.gaussian((1.0, 1.0))) == IF.Algorithm.FIRTiled()
    assert IF.filter_algorithm(v, KernelFactors.IIRGaussian((2.0, 2.0))) == IF.Algorithm.IIR()
    assert IF.filter_algorithm(v, (KernelFactors.IIRGaussian(2.0), IF.centered(np.ones(3)))) == IF.Algorithm.Mixed()


def test_method_errors_and_window_errors():
    r = IF.CPU1(IF.Algorithm.FIR())
    with pytest.raises(IF.MethodError):
        IF.imfilter(r, np.zeros(8), (IF.centered(np.ones(3)),), "replicate", IF.Algorithm.FIR())
    with pytest.raises(IF.ArgumentError):
        IF.imfilter(np.zeros(8), (IF.centered(np.ones(3)),), "inner")
    with pytest.raises(IF.ArgumentError):
        IF.resolve_window(())
    with pytest.raises(RuntimeError):
        IF.resolve_window((3, 4))
    assert IF.resolve_window(5) == (range(-2, 3),)
    assert IF.resolve_window((range(-1, 2), range(0, 1))) == (range(-1, 2), range(0, 1))


def test_explicit_padding_too_small_is_dimension_mismatch():
    A = np.ones((8, 8))
    kern = Kernel.gaussian((1, 1), (3, 3))
    with pytest.raises(IF.ArgumentError):
        IF.imfilter(A, kern, IF.Fill(0, (3,)))
    with pytest.raises(IF.DimensionMismatch):
        IF.imfilter(A, kern, IF.Fill(0, (1, 0)))
    with pytest.raises(IF.DimensionMismatch):
        IF.imfilter(A, kern, IF.Fill(0, (0, 0)))


def test_factorkernel_rank_pretest_agrees_with_svd():
    """factorkernel's quick test only ever rejects kernels the SVD rank test
    rejects: rank one plus perturbations around the tolerance, over scales and
    shapes."""
    import sys
    m = sys.modules["imagefiltering.imfilter"]
    rng = np.random.default_rng(3)
    eps = np.sqrt(np.finfo(np.float64).eps)
    seen = set()
    for shape in ((2, 2), (3, 5), (7, 7), (21, 15)):
        for scale in (1e-7, 1e-3, 1.0, 1e6):
            for level in (0.0, 0.1, 0.9, 1.1, 10.0, 1e3, 1e8):
                a = scale * np.outer(rng.standard_normal(shape[0]), rng.standard_normal(shape[1]))
                e = rng.standard_normal(shape)
                a = a + level * eps * e / np.linalg.norm(e, 2)
                S = np.linalg.svd(a)[1]
                separable = all(s < eps for s in S[1:])
                if m._far_from_rank_one(a):
                    assert not separable
                seen.add((m._far_from_rank_one(a), separable))
    assert (True, False) in seen and (False, True) in seen


# ---- dispatch rules of the library (host functions, no GPU) --------------------------------------
U8, N0F8, F32, F64, BF16, F16 = range(6)  # eltype codes


def test_separable_march_rule():
    """Which equal pairs of factors march down 128-column strips: wide images
    above the size line, by eltype; not narrow ones, whose strips would be half
    empty, in one plane or in a stack."""
    import ctypes as C
    from imagefiltering import _lib
    pays = _lib.load()._ZN3ifm14sep_march_paysEiilll
    pays.argtypes, pays.restype = [C.c_int, C.c_int] + [C.c_int64] * 3, C.c_bool
    for k in (3, 5, 7, 9, 13, 17, 21, 25, 29, 33):
        line = 4_000_000 * max(k, 13) // 13
        for dt in (U8, N0F8, F32, BF16, F16):
            assert not pays(k, dt, 4096, line // 4096 - 1, 1)
            assert pays(k, dt, 4096, 4 * line // 4096, 1)
            assert pays(k, dt, 512, 128, 4 * line // (512 * 128))
            if k > 5 or dt in (BF16, F16):
                assert not pays(k, dt, 60, 4 * line // 60, 1)
                assert not pays(k, dt, 64, 64, 4 * line // 4096)
            # every size above one that marches marches too
            took = [pays(k, dt, 300, line * f // 1200, 1) for f in range(4, 20)]
            assert took == sorted(took)
        assert pays(k, F32, 4096, line // 4096 + 1, 1)
    assert not pays(21, BF16, 4096, 6_500_000 // 4096 + 1, 1)
    assert pays(29, BF16, 4096, 4096, 1) and pays(33, F16, 4096, 4096, 1)


def test_separable_march_rule_of_batches():
    import ctypes as C
    from imagefiltering import _lib
    L = _lib.load()
    shape, line = L._ZN3ifm15sep_march_shapeEiiiill, L._ZN3ifm14sep_march_lineEil
    shape.argtypes, shape.restype = [C.c_int] * 4 + [C.c_int64] * 2, C.c_int
    line.argtypes, line.restype = [C.c_int, C.c_int64], C.c_bool
    NEVER, SLOWER, FASTER = range(3)
    for k in (3, 5, 7, 9, 13, 17, 21, 25, 29, 33):
        px = 16_000_000 * max(k, 13) // 13
        assert not line(k, px - 1) and line(k, px + 1)
        assert shape(k, k, F32, F64, 1024, 1024) == FASTER and shape(k, k, BF16, F64, 1024, 1024) == FASTER
        assert shape(k, k, F64, F64, 1024, 1024) == shape(k, k + 2, F32, F64, 1024, 1024) == NEVER
        for dt in (N0F8, F32, BF16):
            assert shape(k, k, dt, F64, 60, 300) == shape(k, k, dt, F32, 64, 64) == SLOWER
        assert shape(k, k, BF16, BF16, 300, 64) == SLOWER
        if k < 21:
            assert shape(k, k, BF16, BF16, 1000, 1000) == SLOWER
    assert shape(11, 11, F32, F64, 1024, 1024) == NEVER


def test_median_bit_plane_rule():
    """Medians of codes: 5 x 5 and 7 x 7 windows take bit planes where the images
    fill enough 128 x 64 tiles, in one plane or in a stack; not stacks of planes
    that leave the tiles mostly empty, however many."""
    import ctypes as C
    from imagefiltering import _lib
    bits = _lib.load()._ZN3ifm14median_on_bitsEilll
    bits.argtypes, bits.restype = [C.c_int] + [C.c_int64] * 3, C.c_bool
    for k in (3, 9):
        assert bits(k, 9, 9, 1) and bits(k, 24, 24, 2000)
    for k in (5, 7):
        assert not bits(k, 1024, 1024, 1) and bits(k, 1448, 1448, 1) and bits(k, 8192, 8192, 1)
        assert bits(k, 100, 100, 200) and bits(k, 300, 300, 60)
        for planes in (200, 2000, 100000):
            assert not bits(k, 24, 24, planes) and not bits(k, 64, 32, planes)
        assert not bits(k, 64, 64, 300) and not bits(k, 40, 40, 300)
    assert bits(7, 64, 64, 3000) and not bits(5, 64, 64, 3000)


def test_factorkernel_common_kernels(monkeypatch):
    """Kernels in common use that are not of rank one are told apart without the
    SVD; rank-one ones, thin ones and ones with entries that are not finite are
    left to it, whatever their scale."""
    import sys
    m = sys.modules["imagefiltering.imfilter"]
    rng = np.random.default_rng(4)
    y, x = np.mgrid[-5:6, -5:6]
    far = [np.asarray(k.data) for k in (IF.Kernel.LoG(2.0), IF.Kernel.LoG(8.0), IF.Kernel.DoG(2.0))]
    far += [rng.standard_normal((n, n + d)) for n in (2, 3, 7, 21, 45) for d in (0, 1)]
    far += [np.array([[0, 1, 0], [1, -4, 1], [0, 1, 0.0]]), (np.hypot(x, y) <= 5) * 1.0, np.eye(9), np.asfortranarray(rng.random((6, 4)))]
    near = [np.outer(rng.standard_normal(a), rng.standard_normal(b)) * s for a, b in ((2, 2), (3, 5), (7, 7), (21, 21))
            for s in (1e-12, 1e-3, 1.0, 1e9)]
    near += [rng.random((1, 7)), rng.random((7, 1)), np.zeros((5, 5)), np.full((7, 7), np.nan), np.full((4, 4), np.inf)]
    with np.errstate(all="raise"):
        assert not any(m._far_from_rank_one(a) for a in near)
        assert all(m._far_from_rank_one(a) for a in far)
    monkeypatch.setattr(np.linalg, "svd", None)
    for a in far:
        k, = IF.factorkernel(IF.centered(a))
        np.testing.assert_array_equal(np.asarray(k.data), a)


def test_default_algorithm_of_float64_images_is_the_hosts():
    """No library call is made to learn that Float64 pixels are not taken."""
    import sys
    m = sys.modules["imagefiltering.imfilter"]
    img = object.__new__(IF.DeviceArray)
    img.shape, img.eltype, img.order, img._ptr = (100, 90), IF.Float64, "F", None
    kern = (IF.centered(np.random.default_rng(0).random((9, 9))),)
    assert m._run_default(None, img, kern, IF.borderinstance("reflect")) is False
