"""The LDS-tiled GEMM (gemm_f32_tile) and the small-M GEMM (gemm_f32_ksplit) at
the sizes and operand values where their two paths, fp16 pairs and plain fp32
products, meet: K around a panel and around the fp16 path's least K, ragged
tiles of every form, every orientation, and operands below, above and outside
fp16's range. Which kernel the shapes run on 256 CUs is checked, without a GPU, by
test_gemm_plan.py."""
import ctypes as C

import numpy as np
import pytest

from inferc_amd import lib as L
from inferc_amd.rt import Context, Tensor

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with Context(0) as c:
        yield c


def _run(ctx, a, b, ta, tb, c=None):
    """Y = op(A) op(B) (+ row C) for op(A) [M, K], op(B) [K, N] in numpy."""
    (M, K), N = a.shape, b.shape[1]
    A = Tensor.from_numpy(ctx, np.ascontiguousarray(a.T if ta else a))
    B = Tensor.from_numpy(ctx, np.ascontiguousarray(b.T if tb else b))
    Cd = Tensor.from_numpy(ctx, c) if c is not None else None
    Y = Tensor.empty(ctx, (M, N))
    L.check(ctx._lib.inferc_hip_gemm_f32(
        ctx.handle, ta, tb, M, N, K, C.c_float(1.0), A.ptr, A.shape[1], B.ptr, B.shape[1],
        C.c_float(1.0), Cd.ptr if Cd else None, L.C_ROW if Cd else L.C_NONE, 0, None, 0,
        L.ACT_NONE, Y.ptr, N))
    return Y.numpy()


def _check(got, a, b):
    """Against 64 bits, relative to S = sum |a| |b|: an fp16 pair is within 2^-23 of
    its value and the product of two low halves within 2^-22 of the product; what fp16
    cannot hold of small elements is bounded by K 2^-23 S, the rounding of a sum of K in
    fp32 by K 2^-24 S; and K times half a subnormal step (2^-149) where the sums are that small."""
    a, b = a.astype(np.float64), b.astype(np.float64)
    K = a.shape[1]
    mag = np.abs(a) @ np.abs(b)
    lim = (2.0 ** -21 + 3 * K * 2.0 ** -24) * mag + K * 2.0 ** -150
    err = np.abs(got - a @ b)
    assert (err <= lim).all(), float((err / np.maximum(lim, 1e-300)).max())


# M > 512 keeps the small-M kernel away; the tile forms' edges are 64 and 128
EDGES_64 = [(513, 1, 1), (513, 65, 31), (576, 63, 32), (640, 129, 33), (515, 64, 63),
            (520, 68, 64), (519, 130, 65), (1000, 257, 96), (513, 384, 1536), (514, 131, 1601),
            (4097, 1025, 68), (4100, 1100, 40), (70, 40001, 65), (40000, 66, 96),
            (516, 64, 4), (600, 132, 12), (1000, 260, 28), (2600, 1200, 24)]
EDGES_128 = [(5120, 1280, 128), (2000, 2000, 130), (1921, 2047, 1), (2047, 1921, 31),
             (2001, 1999, 45), (1990, 2011, 63), (1985, 1985, 64), (2033, 1987, 97),
             (100, 50257, 40), (2000, 2000, 20)]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", EDGES_64 + EDGES_128)
def test_gemm_tile_edges(ctx, ta, tb, M, N, K):
    rng = np.random.default_rng(M * 7 + N * 3 + K + 2 * ta + tb)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = (0.02 * rng.standard_normal((K, N))).astype(np.float32)
    _check(_run(ctx, a, b, ta, tb), a, b)


# M <= 512 with whole float4 rows: every form of the small-M kernel (16x16,
# 16x32, 16x48 over two blocks, 32x64, 32x48) and the tiles that replace it
# from two or three rounds of blocks up
SMALL = [(2, 4, 4), (33, 64, 60), (127, 2304, 60), (120, 1732, 36), (31, 768, 64),
         (64, 2304, 132), (17, 132, 68), (17, 132, 420), (97, 772, 100), (97, 772, 708),
         (130, 1540, 96), (130, 1732, 96), (128, 768, 3072), (100, 768, 2052), (127, 2304, 288),
         (255, 2304, 288), (129, 3072, 772), (300, 2308, 768), (259, 2308, 100), (130, 4100, 772),
         (512, 3072, 768), (131, 768, 2048), (200, 60, 2052)]


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", SMALL)
def test_gemm_small_m_edges(ctx, tb, M, N, K):
    rng = np.random.default_rng(M * 7 + N * 3 + K + tb)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = (0.02 * rng.standard_normal((K, N))).astype(np.float32)
    _check(_run(ctx, a, b, 0, tb), a, b)


# few tiles: K goes over as many blocks as there are CUs, in splits of 192 at least
@pytest.mark.parametrize("ta,tb,M,N,K", [
    (0, 0, 1, 3, 575), (0, 0, 1, 3, 576), (0, 0, 64, 63, 1500), (1, 0, 100, 200, 1501),
    (0, 0, 600, 256, 1000), (0, 1, 513, 129, 2049), (1, 1, 512, 512, 769), (0, 0, 65, 63, 20000)])
def test_gemm_few_tiles_split_k(ctx, ta, tb, M, N, K):
    rng = np.random.default_rng(M + N + K)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = (0.02 * rng.standard_normal((K, N))).astype(np.float32)
    c = rng.standard_normal(N).astype(np.float32)
    got = _run(ctx, a, b, ta, tb, c)
    # (the sum with C rounds once more, at 2^-24 of an output)
    err = np.abs(got - (a.astype(np.float64) @ b + c))
    mag = np.abs(a).astype(np.float64) @ np.abs(b) + np.abs(c)
    assert (err <= (2.0 ** -21 + 3 * K * 2.0 ** -24) * mag).all()
    np.testing.assert_array_equal(_run(ctx, a, b, ta, tb, c), got)


RANGES = [(600, 200, 192), (4224, 1100, 100), (70, 200, 384), (128, 768, 3072),
          (2000, 2010, 100)]
VALUES = ["tiny_a", "tiny_b", "zero_row", "late_row", "huge", "mixed", "subnormal", "integers",
          "one_hot"]


@pytest.mark.parametrize("kind", VALUES)
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", RANGES)
def test_gemm_tile_operand_ranges(ctx, M, N, K, kind, tb):
    rng = np.random.default_rng(len(kind) * 31 + M)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = (0.02 * rng.standard_normal((K, N))).astype(np.float32)
    if kind == "tiny_a":
        a *= np.float32(1e-12)
    elif kind == "tiny_b":
        b *= np.float32(1e-9)
    elif kind == "zero_row":
        a[::37] = 0.0
        b[:, ::41] = 0.0
    elif kind == "late_row":  # a row whose first panel is zero and the rest small
        a[::37, :32] = 0.0
        a[::37, 32:] *= np.float32(1e-7)
    elif kind == "huge":  # beyond fp16
        a[5, K // 2] = 1e20
        b[K - 1, 7] = -7e4
    elif kind == "mixed":  # every row and column spans many decades
        a *= np.float32(10.0) ** rng.uniform(-8, 3, a.shape).astype(np.float32)
        b *= np.float32(10.0) ** rng.uniform(-6, 3, b.shape).astype(np.float32)
    elif kind == "subnormal":
        a[3] = np.float32(1e-41)
        b[:, 2] = np.float32(3.0)
    elif kind == "integers":
        a = rng.integers(-30, 31, a.shape).astype(np.float32)
        b = rng.integers(-30, 31, b.shape).astype(np.float32)
    elif kind == "one_hot":
        a = np.eye(M, K, dtype=np.float32)
        a[K:, 0] = 1.0
    got = _run(ctx, a, b, 0, tb)
    _check(got, a, b)
    if kind in ("integers", "one_hot"):  # exact in fp32 whatever the order
        np.testing.assert_array_equal(got, (a.astype(np.float64) @ b).astype(np.float32))


MEETS = [(128, 768, 768), (600, 200, 768), (2, 64, 128), (4000, 3072, 96), (77, 50257, 96)]


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("M,N,K", MEETS)
@pytest.mark.parametrize("pattern", ["block", "checker", "late", "columns"])
def test_gemm_large_elements_meet_zeros(ctx, tb, M, N, K, pattern):
    """Outputs made of small elements alone, beside large ones that meet zeros of the
    other operand: as exact as any fp32 sum (5e-7 in the 2-norm at K = 768; 2e-6 is
    asked), however small."""
    rng = np.random.default_rng(M + N)
    h = N // 2
    for s in (1e-3, 1e-5, 1e-7, 1e-9, 1e-12, 1e-25):
        a = rng.standard_normal((M, K))
        b = 0.02 * rng.standard_normal((K, N))
        part = (slice(None), slice(h, None))  # the outputs made of small elements
        if pattern == "block":  # b's two blocks see 16 large and K - 16 small columns of a
            a[:, 16:] *= s
            b[16:, :h] = 0.0
            b[:16, h:] = 0.0
        elif pattern == "checker":  # the same, by turns over rows and columns
            big = np.arange(K) % 2 == 0
            a[0::2, big] *= s
            a[1::2, ~big] *= s
            b[np.ix_(big, np.arange(N) % 2 == 0)] = 0.0
            b[np.ix_(~big, np.arange(N) % 2 == 1)] = 0.0
            part = (slice(0, None, 2), slice(1, None, 2))
        elif pattern == "late":  # the large ones come after the first panel
            a[:, :64] *= s
            b[64:, h:] = 0.0
        else:  # small and large elements of b
            b[:, h:] *= s
            b[16:24, h:] = 1.0
            a[:, 16:24] = 0.0
        a, b = a.astype(np.float32), b.astype(np.float32)
        ref = (a.astype(np.float64) @ b)[part]
        got = _run(ctx, a, b, 0, tb)[part]
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert err <= 2e-6, (s, err)


@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("M,N,K", [(600, 200, 768), (2000, 2003, 512), (4000, 3072, 512),
                                   (128, 768, 768)])
def test_gemm_zero_rows_that_stay_zero_or_not(ctx, M, N, K, ta):
    """Rows of A and columns of B that are zero over the first panel: over all of K, or
    with one element near the end (in the tiles, the former keep the fp16 path and the
    latter leave it on the way)."""
    rng = np.random.default_rng(K)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = (0.02 * rng.standard_normal((K, N))).astype(np.float32)
    a[::5] = 0.0
    b[:, ::7] = 0.0
    _check(_run(ctx, a, b, ta, 0), a, b)
    a[10, K - 40] = 3e-9
    b[K - 35, 14] = -5e-8
    got = _run(ctx, a, b, ta, 0)
    _check(got, a, b)
    want = a[10, K - 40].astype(np.float64) * b[K - 40]
    assert np.abs(got[10] - want).max() <= 2.0 ** -22 * np.abs(want).max()


INFINITIES = [(0, 0, 777, 333, 160), (1, 1, 777, 333, 160), (0, 1, 500, 332, 160),
              (0, 1, 500, 332, 288), (0, 0, 500, 332, 160), (0, 0, 2000, 2003, 160),
              (0, 1, 2000, 2003, 160), (1, 0, 2000, 2003, 160)]


@pytest.mark.parametrize("ta,tb,M,N,K", INFINITIES)
def test_gemm_tile_infinities_and_nan(ctx, ta, tb, M, N, K):
    """(500 rows: the small-M kernel, with B transposed from K = 260; 2000 rows: 128x128
    tiles)"""
    rng = np.random.default_rng(9)
    a = rng.standard_normal((M, K)).astype(np.float32)
    b = rng.standard_normal((K, N)).astype(np.float32)
    a[3, 17], a[130, 159], a[400, 0] = np.inf, -np.inf, np.nan
    b[80, 64], b[2, 300] = np.inf, np.finfo(np.float32).max
    b[17, 5] = 0.0  # inf * 0
    c = rng.standard_normal(N).astype(np.float32)
    got = _run(ctx, a, b, ta, tb, c)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = (a.astype(np.float64) @ b.astype(np.float64) + c).astype(np.float32)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    np.testing.assert_array_equal(np.isinf(got), inf)
    np.testing.assert_array_equal(got[inf], ref[inf])
    ok = np.isfinite(ref) & (np.abs(ref) < 1e30)
    assert np.abs(got[ok] - ref[ok]).max() <= 1e-3


@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("K,lim", [(64, 8.7e-8), (128, 9.2e-8), (256, 1.0e-7)])
def test_small_m_one_group_rounding(ctx, K, lim, tb):
    """K up to 256 is eight sums of at most 32 products in the 16-row blocks: over half-zero
    rows 8.0e-8, 8.5e-8 and 9.4e-8 in the 2-norm with exact operands, where pairs (rounded
    at 2^-24 each) come to 9.4e-8, 9.9e-8 and 1.06e-7."""
    for M, N in [(32, 768), (300, 300)]:
        rng = np.random.default_rng(K + M)
        a = np.maximum(rng.standard_normal((M, K)), 0).astype(np.float32)
        b = (0.02 * rng.standard_normal((K, N))).astype(np.float32)
        ref = a.astype(np.float64) @ b
        assert np.linalg.norm(_run(ctx, a, b, 0, tb) - ref) <= lim * np.linalg.norm(ref)


EPILOGUES = [(530, 70, 96), (4200, 1000, 96), (2000, 1990, 96), (1990, 2001, 40)]


def test_gemm_tile_residual_c_and_activation(ctx):
    """The epilogue over ragged tiles of every form: full C, residual, GELU."""
    from math import erf
    for M, N, K in EPILOGUES:
        rng = np.random.default_rng(M)
        a = rng.standard_normal((M, K)).astype(np.float32)
        b = (0.1 * rng.standard_normal((K, N))).astype(np.float32)
        c = rng.standard_normal((M, N)).astype(np.float32)
        r = rng.standard_normal((M, N)).astype(np.float32)
        A, B, Cd, R = (Tensor.from_numpy(ctx, x) for x in (a, b, c, r))
        Y = Tensor.empty(ctx, (M, N))
        L.check(ctx._lib.inferc_hip_gemm_f32(
            ctx.handle, 0, 0, M, N, K, C.c_float(0.5), A.ptr, K, B.ptr, N, C.c_float(2.0), Cd.ptr,
            L.C_FULL, N, R.ptr, N, L.ACT_GELU_ERF, Y.ptr, N))
        v = 0.5 * (a.astype(np.float64) @ b) + 2.0 * c + r
        rows = rng.integers(0, M, 64)
        ref = v[rows] * 0.5 * (1.0 + np.vectorize(erf)(v[rows] / np.sqrt(2.0)))
        assert np.abs(Y.numpy()[rows] - ref).max() <= 2e-5
