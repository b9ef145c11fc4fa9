"""fp32 GEMMs on the bf16 matrix cores (mgc_hip_gemm_planes) against float64.

Every tile shape is pinned through mgc_hip_gemm_args.kernel at the edges of its tiles (128 or 32
rows, 32 to 128 columns, 32 k per stage, 16 k per MFMA, eight waves sharing K), for row-major A, also
of rows that are only 4-byte aligned (K no multiple of four), NHWC convolutions and a concatenated K, with a K split and a rotating epilogue. The tolerance is the standard bound of a
summation: with S = sum |a||b| of an element, at most 6 K / 16 + 8 roundings of 2^-24 S for the MFMA
accumulations and the epilogue, and 2^-23 S for the products the split drops.

Operands the split cannot carry are recomputed in fp32: infinities and NaN come out as float
arithmetic has them, rows or columns below 2^-95 keep fp32 precision.
"""

from __future__ import annotations

import ctypes
import time

import numpy as np
import pytest

from capi import ACTS, MGC_ERR_ARGS, MGC_OK, MGC_OP_CONV_NHWC, GemmArgs, Hip, bind
from ml_graph_compiler.codegen.build import load_kernel_library
from oracle import interpreter as oracle

pytestmark = pytest.mark.gpu

FAMILIES = {"128x128": 8, "128x64": 9, "32x64": 10, "32x32": 11}


class Runner:
    def __init__(self) -> None:
        self.lib = load_kernel_library()
        bind(self.lib)
        self.lib.mgc_hip_gemm_make_planes.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_long, ctypes.c_int,
                                                      ctypes.c_int, ctypes.c_void_p]
        self.lib.mgc_hip_gemm_planes.argtypes = [ctypes.c_void_p] * 3
        self.hip = Hip()
        self.x = self.lib.mgc_hip_exec_create(None)
        assert self.x, self.lib.mgc_hip_last_error()

    def planes(self, b: np.ndarray) -> tuple[int, int]:
        """Device addresses of b ([N][K]) and of its planes."""
        n, k = b.shape
        pb = self.hip.upload(b)
        planes = self.hip.alloc((n + 31) // 32 * 32 * ((k + 31) // 32 * 32) * 6 + (n + 31) // 32 * 32 + 256)
        self.lib.mgc_hip_gemm_make_planes(self.x, pb, k, n, k, planes)
        return pb, planes

    def run(self, g: GemmArgs, planes: int) -> int:
        self.lib.mgc_hip_gemm_planes(self.x, ctypes.byref(g), planes)
        return self.lib.mgc_hip_exec_status(self.x)

    def gemm(self, family: str, a: np.ndarray, b: np.ndarray, fill=None, split: int = 1, m: int | None = None,
             bias=None, bias_mode=0, res=None, alpha=1.0, beta=1.0, act="none", lo=-0.5, hi=0.75) -> np.ndarray:
        m = a.shape[0] if m is None else m
        n, k = b.shape
        g = GemmArgs()
        g.M, g.N, g.K = m, n, k
        g.a.p, g.a.rs, g.a.cs = self.hip.upload(a), k, 1
        g.b.rs, g.b.cs = 1, k
        g.b.p, planes = self.planes(b)
        g.c, g.ldc = self.hip.empty(4 * m * n), n
        g.alpha, g.beta, g.bias_mode = alpha, beta, bias_mode
        g.bias = self.hip.upload(bias) if bias is not None else None
        if res is not None:
            g.res, g.ldr = self.hip.upload(res), n
        g.act, g.lo, g.hi = ACTS.index(act), lo, hi
        g.kernel, g.split_k = FAMILIES[family], split
        if split > 1:
            g.workspace, g.workspace_floats = self.hip.empty(4 * split * m * n), split * m * n
        if fill is not None:
            fill(g)
        code = self.run(g, planes)
        assert code == MGC_OK, (code, self.lib.mgc_hip_last_error())
        out = self.hip.download(g.c, (m, n))
        self.hip.free()
        return out


@pytest.fixture(scope="module")
def runner():
    r = Runner()
    yield r
    r.lib.mgc_hip_exec_destroy(r.x)


def _bound(a64: np.ndarray, b64: np.ndarray, k: int) -> np.ndarray:
    s = np.abs(a64) @ np.abs(b64).T
    return (6 * k / 16 + 10) * 2.0**-24 * s


def _check(got, a64, b64, bias=None, bias_mode=0, res=None, alpha=1.0, beta=1.0, act="none"):
    y = alpha * (a64 @ b64.T)
    scale = abs(alpha) * _bound(a64, b64, a64.shape[1])
    # the epilogue's own roundings (alpha, bias, beta, residual: four of 2^-24) are of partial sums,
    # whose size the terms' sizes bound where they cancel in y
    terms = np.abs(y)
    if bias_mode:
        b = bias[None, :] if bias_mode == 1 else bias[:, None]
        y, terms = y + b.astype(np.float64), terms + np.abs(b)
    if res is not None:
        y, terms = y + beta * res.astype(np.float64), terms + np.abs(beta * res)
    scale = scale + 2.0**-22 * terms + 1e-30
    if act != "none":
        y = oracle.activation(y, {"activation": act, "clip_min": -0.5, "clip_max": 0.75})
        scale = 1.2 * scale + 5e-7  # slope at most 1.13 (GELU), the activations' own approximation
    assert np.all(np.abs(got - y) <= scale), float(np.max(np.abs(got - y) / scale))


# rows of K % 4 have no 32 x 64 form (32 x 32 tiles run instead)
@pytest.mark.parametrize("family,k", [(f, k) for k in (4, 16, 28, 32, 36, 64, 68, 100, 260, 1028, 5, 7, 30, 33, 65, 99, 259)
                                      for f in FAMILIES if f != "32x64" or k % 4 == 0])
def test_shapes(runner, family, k):
    """Rows and columns at the tiles' edges, K at the stages', every epilogue and K splits."""
    rng = np.random.default_rng(k)
    for i, (m, n) in enumerate([(1, 1), (31, 33), (127, 63), (128, 64), (129, 65), (130, 127), (200, 128), (257, 129), (64, 260)]):
        a = rng.standard_normal((m, k)).astype(np.float32)
        b = (rng.standard_normal((n, k)) * 0.1).astype(np.float32)
        mode = i % 3
        bias = rng.standard_normal((0, n, m)[mode]).astype(np.float32) if mode else None
        res = rng.standard_normal((m, n)).astype(np.float32) if i % 2 else None
        ep = {"bias": bias, "bias_mode": mode, "res": res, "alpha": 0.5 if i % 4 == 3 else 1.0, "beta": -0.75, "act": ACTS[(i + k) % 7]}
        split = (1, 2, 3)[i % 3] if k >= 64 else 1
        got = runner.gemm(family, a, b, split=split, **ep)
        _check(got, a.astype(np.float64), b.astype(np.float64), **ep)


def _split(x: np.ndarray) -> list[np.ndarray]:
    """The three bf16 parts of floats, largest first, in float64."""
    parts, rest = [], x.astype(np.float32)
    for _ in range(3):
        bits = rest.view(np.uint32)
        part = ((bits + 0x7FFF + ((bits >> 16) & 1)) & np.uint32(0xFFFF0000)).view(np.float32)  # nearest, ties to even
        parts.append(part.astype(np.float64))
        rest = rest - part
    assert not rest.any()
    return parts


@pytest.mark.parametrize("family", FAMILIES)
@pytest.mark.parametrize("k", [96, 99, 512, 540, 1056, 1060, 2076])
def test_every_product_of_the_split(runner, family, k):
    """Sums of four products in a long K, spread over the stages, their halves and a last partial stage: few
    enough roundings to see any one of the six bf16 products missing anywhere. A leading sum and the
    corrections round at most twice 2^-24 of the sum per product and once where they meet, and the
    dropped products are 2^-25: 10 x 2^-24 S. K of 512 and more runs the main loop with the written-out order,
    for the small tiles every wave's share of K."""
    rng = np.random.default_rng(k)
    m, n, t = 140, 136, 4
    for sparse_a in (True, False):
        shape, dense = ((m, k), (n, k)) if sparse_a else ((n, k), (m, k))
        thin = np.zeros(shape, np.float32)
        at = np.stack([rng.permutation(k)[:t] for _ in range(shape[0])])
        at[: shape[0] // 2, 0] = k - 1 - np.arange(shape[0] // 2) % 36  # the last stage and the one before
        np.put_along_axis(thin, at, rng.uniform(1.0, 2.0, at.shape).astype(np.float32), 1)
        full = (rng.uniform(1.0, 2.0, dense) * rng.choice([-1.0, 1.0], dense)).astype(np.float32)
        a, b = (thin, full) if sparse_a else (full, thin)
        got = runner.gemm(family, a, b)
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        bound = 10 * 2.0**-24 * (np.abs(a64) @ np.abs(b64).T)
        assert np.all(np.abs(got - a64 @ b64.T) <= bound)
        pa, pb = _split(a), _split(b)
        for i, j in ((0, 0), (0, 1), (1, 0), (0, 2), (1, 1), (2, 0)):  # what the bound sees
            lost = np.abs(pa[i] @ pb[j].T)
            assert np.mean(lost > 2 * bound) > 0.02, (i, j)


@pytest.mark.parametrize("family", FAMILIES)
@pytest.mark.parametrize("k", [36, 516])
def test_rows_of_four_byte_alignment(runner, family, k):
    """K a multiple of four, A four bytes off the 16-byte alignment."""
    rng = np.random.default_rng(k)
    a = rng.standard_normal((130, k)).astype(np.float32)
    b = (rng.standard_normal((70, k)) * 0.1).astype(np.float32)

    def fill(g):
        g.a.p = runner.hip.upload(np.concatenate([[np.float32(np.nan)], a.ravel()])) + 4

    _check(runner.gemm(family, a, b, fill=fill), a.astype(np.float64), b.astype(np.float64))


def _im2col(x: np.ndarray, kh: int, stride: int, pad: int) -> np.ndarray:
    n, h, w, c = x.shape
    xp = np.pad(x, ((0, 0), (pad, pad), (pad, pad), (0, 0)))
    oh, ow = (h + 2 * pad - kh) // stride + 1, (w + 2 * pad - kh) // stride + 1
    cols = [xp[:, i : i + stride * (oh - 1) + 1 : stride, j : j + stride * (ow - 1) + 1 : stride] for i in range(kh) for j in range(kh)]
    return np.stack(cols, 3).reshape(n * oh * ow, kh * kh * c)


@pytest.mark.parametrize("family", FAMILIES)
@pytest.mark.parametrize("c,kh,stride,pad,hw", [(8, 3, 1, 1, 9), (8, 3, 2, 0, 15), (24, 3, 1, 1, 7), (64, 3, 1, 1, 12), (64, 1, 2, 0, 14), (40, 5, 2, 2, 11)])
def test_convolutions(runner, family, c, kh, stride, pad, hw):
    _convolution(runner, family, c, kh, stride, pad, hw)


@pytest.mark.parametrize("family", FAMILIES)
@pytest.mark.parametrize("c,kh,stride,pad,hw,split", [(32, 3, 1, 1, 9, 1), (32, 3, 2, 0, 11, 4), (96, 3, 2, 1, 9, 3), (64, 3, 1, 2, 6, 5), (160, 2, 1, 1, 5, 2)])
def test_convolutions_one_tap_per_stage(runner, family, c, kh, stride, pad, hw, split):
    """Channels in multiples of 32: a K stage reads one window tap; K splits start inside a tap's
    channels (32 of 64 or 96) and at taps, the last part shorter or empty."""
    _convolution(runner, family, c, kh, stride, pad, hw, split)


def _convolution(runner, family, c, kh, stride, pad, hw, split=1):
    rng = np.random.default_rng(c + kh)
    x = rng.standard_normal((3, hw, hw, c)).astype(np.float32)
    cols = _im2col(x, kh, stride, pad)
    m, k = cols.shape
    n = 70
    b = (rng.standard_normal((n, k)) * 0.1).astype(np.float32)
    o = (hw + 2 * pad - kh) // stride + 1

    def fill(g):
        g.a.kind, g.a.p = MGC_OP_CONV_NHWC, runner.hip.upload(x)
        g.a.H = g.a.W = hw
        g.a.C = g.a.cg = c
        g.a.KH = g.a.KW = kh
        g.a.SH = g.a.SW = stride
        g.a.DH = g.a.DW = 1
        g.a.PT = g.a.PL = pad
        g.a.OH = g.a.OW = o

    got = runner.gemm(family, x, b, fill=fill, m=m, split=split, act="relu")
    _check(got, cols.astype(np.float64), b.astype(np.float64), act="relu")


@pytest.mark.parametrize("family", FAMILIES)
def test_concatenated_k(runner, family):
    """Columns past k1 come from an image sampled at a stride (a projection shortcut)."""
    rng = np.random.default_rng(5)
    nb, hw, c2, k1, n = 2, 9, 36, 64, 100
    o = (hw + 1) // 2
    x = rng.standard_normal((nb, hw, hw, c2)).astype(np.float32)
    a = rng.standard_normal((nb * o * o, k1)).astype(np.float32)
    whole = np.concatenate([a, x[:, ::2, ::2].reshape(-1, c2)], axis=1)
    b = (rng.standard_normal((n, k1 + c2)) * 0.1).astype(np.float32)

    def fill(g):
        g.a.rs, g.k1 = k1, k1
        g.a2.kind, g.a2.p = MGC_OP_CONV_NHWC, runner.hip.upload(x)
        g.a2.H = g.a2.W = hw
        g.a2.C = g.a2.cg = c2
        g.a2.KH = g.a2.KW = g.a2.DH = g.a2.DW = 1
        g.a2.SH = g.a2.SW = 2
        g.a2.OH = g.a2.OW = o

    got = runner.gemm(family, a, b, fill=fill)
    _check(got, whole.astype(np.float64), b.astype(np.float64))


@pytest.mark.parametrize("family", FAMILIES)
@pytest.mark.parametrize("k", [96, 99, 544, 1060])
def test_values_the_split_cannot_carry(runner, family, k):
    """Infinities, NaN, overflow and the largest floats as fp32 has them; tiny rows and columns to
    fp32 precision; zeros exact; everything else in the same tiles untouched."""
    rng = np.random.default_rng(9)
    m, n = 140, 72
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.choice([0.5, -2.0, 1.0, 0.25, -1.5], (n, k)).astype(np.float32)  # exact in bf16: zero low parts
    a[3, 5] = np.inf
    a[4, 6] = -np.inf
    a[5, 7] = np.nan
    a[6, 8], a[6, 9] = np.inf, -np.inf
    a[7, 10] = 3.4e38
    a[8] = 0.0
    a[9] *= np.float32(2.0**-120)
    a[130] *= np.float32(2.0**-100)
    b[11, 3] = np.inf
    b[11, 10] = 0.5  # a[7, 10] times it is finite: an overflow and an infinity of other signs are NaN in one order only
    b[12] *= np.float32(2.0**-118)
    got = runner.gemm(family, a, b)
    with np.errstate(all="ignore"):
        # small whole steps of the exact sum, then rounded to float: infinities and NaN as float has them
        want = (a.astype(np.float64) @ b.astype(np.float64).T).astype(np.float32)
        bound = _bound(np.where(np.isfinite(a), a, 0).astype(np.float64), np.where(np.isfinite(b), b, 0).astype(np.float64), k)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(want))
    np.testing.assert_array_equal(np.isneginf(got), np.isneginf(want))
    ok = np.isfinite(want)
    assert np.all(np.abs(got[ok].astype(np.float64) - want[ok]) <= 4 * bound[ok] + 2.0**-148)
    assert np.all(got[8][np.isfinite(b).all(1)] == 0.0)


@pytest.mark.parametrize("family", FAMILIES)
@pytest.mark.parametrize("k", [96, 99, 544])
def test_small_numbers_beside_normal_ones(runner, family, k):
    """Rows and columns that mix normal numbers with ones down to the smallest subnormal: where the other
    operand is zero at the normal ones, the small ones are the whole sum, and it has fp32 precision.
    The last term: up to eight waves' parts and their seven sums round to a subnormal's 2^-150 each (a
    chain of fp32 products would at every k)."""
    rng = np.random.default_rng(k)
    m, n = 140, 72
    a, b = rng.standard_normal((m, k)), rng.standard_normal((n, k))
    half = rng.permutation(k) < k // 2
    small = 2.0 ** rng.integers(-146, -104, (max(m, n), 1))  # one size to a row: nothing larger hides a loss
    a[:70] = np.where(half, a[:70], a[:70] * small[:70])  # normal at `half`, small elsewhere
    a[70:, half] = 0.0
    b[:36, half] = 0.0
    b[36:] = np.where(half, b[36:], b[36:] * small[36:n])
    a, b = a.astype(np.float32), b.astype(np.float32)
    assert np.any((a != 0) & (np.abs(a) < 2.0**-134)) and np.any((b != 0) & (np.abs(b) < 2.0**-134))
    got = runner.gemm(family, a, b)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want = a64 @ b64.T
    assert np.all(np.abs(got - want) <= _bound(a64, b64, k) + 15 * 2.0**-150)
    assert np.median(np.abs(want[:70, :36])) < 2.0**-100 and np.median(np.abs(want[70:, 36:])) < 2.0**-60


def test_a_matrix_of_nan_costs_no_more_than_fp32_products(runner):
    """Sums that are not finite are computed again, by the whole tile on the fp32 matrix cores: a product of
    NaN alone takes a few times the finite one's time (six bf16 products cost 3/8 of the fp32 ones'), not
    a serial loop's per element."""
    m, n, k = 2048, 3072, 768
    rng = np.random.default_rng(2)
    b = rng.standard_normal((n, k)).astype(np.float32)
    g = GemmArgs()
    g.M, g.N, g.K, g.alpha = m, n, k, 1.0
    g.a.rs, g.a.cs = k, 1
    g.b.rs, g.b.cs = 1, k
    g.b.p, planes = runner.planes(b)
    g.c, g.ldc, g.kernel, g.split_k = runner.hip.empty(4 * m * n), n, FAMILIES["128x128"], 1
    times = []
    for a in (rng.standard_normal((m, k)).astype(np.float32), np.full((m, k), np.nan, np.float32)):
        g.a.p = runner.hip.upload(a)
        best = np.inf
        for _ in range(5):
            t = time.perf_counter()
            assert runner.run(g, planes) == MGC_OK
            best = min(best, time.perf_counter() - t)
        times.append(best)
    runner.hip.free()
    print(f"2048 x 768 x 3072: finite {1e6 * times[0]:.0f} us, NaN {1e6 * times[1]:.0f} us", flush=True)
    assert times[1] < 8 * times[0]


def test_refusals(runner):
    """The families need planes and an A they can read; mgc_hip_gemm has none."""
    a, b = np.ones((128, 32), np.float32), np.ones((64, 32), np.float32)
    g = GemmArgs()
    g.M, g.N, g.K, g.alpha = 128, 64, 32, 1.0
    g.a.p, g.a.rs, g.a.cs = runner.hip.upload(a), 32, 1
    g.b.rs, g.b.cs = 1, 32
    g.b.p, planes = runner.planes(b)
    g.c, g.ldc, g.kernel = runner.hip.empty(4 * 128 * 64), 64, 9
    runner.lib.mgc_hip_gemm(runner.x, ctypes.byref(g))
    assert runner.lib.mgc_hip_exec_status(runner.x) == MGC_ERR_ARGS
    g.M, g.a.p = 127, g.a.p + 4  # only 4-byte aligned: read element-aligned
    assert runner.run(g, planes) == MGC_OK
    g.a.cs, g.a.rs, g.M = 4, 1, 8  # columns apart: refused when pinned, fp32 kernels otherwise
    assert runner.run(g, planes) == MGC_ERR_ARGS
    g.kernel = 0
    assert runner.run(g, planes) == MGC_OK
    runner.hip.free()
