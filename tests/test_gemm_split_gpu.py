"""Products as three-part splits (kernels/split3.h): f32 operands as three bf16
parts each, six part products on the bf16 matrix instruction. Every operand layout,
edges and k tails against float64; infinities, NaN, values whose bf16 rounding
overflows and subnormals, which the split cannot carry and the kernels recompute;
and the error against the f32 instruction's. Of the large sizes below, the
256-row kernel (kernels/gemm_split.h) runs [4097, 32] x [32, 3071] and K = 16384 of the
error test, the walk of 64 x 64 tiles (kernels/gemm.h) the others; the 256-row kernel's
own sizes are in test_gemm_kernels_gpu.py, by the kernel's name.

Bound: a sum of K products in f32 is within K u sum |a||b| of the exact one in any
order (u = 2^-24); the split's 12 roundings per 16 k are fewer than K, and the part
products it leaves out are below 2^-24 |a||b| each, so (K + 2) u sum |a||b| holds."""
import ctypes

import numpy as np
import pytest

from parity import dev, fetch, out
from test_block_ops_gpu import gemm_desc

pytestmark = pytest.mark.gpu


def product(vh, a, b, akc, bkc, off=0, **kw):
    """vh_gemm of a [M, K] and b [K, N] stored k- or row-contiguous, `off` floats into
    their buffers; C has a guard row after it that must come back untouched."""
    M, K = a.shape
    N = b.shape[1]
    pad = np.zeros(off, np.float32)
    A = dev(vh, np.concatenate([pad, (a if akc else a.T).reshape(-1)]))
    B = dev(vh, np.concatenate([pad, (b.T if bkc else b).reshape(-1)]))
    C = dev(vh, np.full((M + 1, N), 7.0, np.float32))
    d = gemm_desc(vh, M, N, K, A.ptr + 4 * off, K if akc else 1, 1 if akc else M, B.ptr + 4 * off, 1 if bkc else N,
                  K if bkc else 1, C.ptr, N, **kw)
    vh.check(vh.lib.vh_gemm(ctypes.byref(d), None))
    path = vh.lib.vh_gemm_last_path()
    got = fetch(vh, C, (M + 1, N))
    np.testing.assert_array_equal(got[M], 7.0)
    return got[:M], path


LAYOUTS = [(True, True), (True, False), (False, True), (False, False)]
#   M, N, K, floats off 16-byte alignment
SIZES = [
    (256, 192, 1366, 0),    # whole 64 x 64 tiles, k tail of 22
    (257, 193, 1361, 1),    # one row and one column past a tile, k tail of 17
    (1000, 777, 1007, 3),   # ragged, k tail of 15
    (4097, 3071, 32, 0),    # 256-row tiles of two k tiles, the round left whole
    (300, 500, 16385, 0),   # past the 256-row kernel's single-chain limit
]


@pytest.mark.parametrize("size", SIZES, ids=str)
@pytest.mark.parametrize("akc,bkc", LAYOUTS)
def test_split_product_sizes(vh, akc, bkc, size):
    M, N, K, off = size
    print("split", size, akc, bkc, flush=True)
    r = np.random.default_rng(M + N + K)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    got, path = product(vh, a, b, akc, bkc, off)
    assert path == vh.GEMM_PATH_PERSISTENT
    ref = a.astype(np.float64) @ b.astype(np.float64)
    bound = (K + 2) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    assert np.all(np.abs(got - ref) <= bound)
    again, _ = product(vh, a, b, akc, bkc, off)
    np.testing.assert_array_equal(again, got)


@pytest.mark.parametrize("akc,bkc", LAYOUTS)
def test_split_product_special_values(vh, akc, bkc):
    """Each special value where the f32 instruction (the WIDE engine) puts it; the
    other elements within the bound of their own exact sums."""
    print("split specials", akc, bkc, flush=True)
    M, N, K = 520, 400, 700
    r = np.random.default_rng(3)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    a[5, 17] = np.inf
    a[6, 699] = -np.inf
    a[300, 0] = np.nan
    a[301, 3] = -3.4e38  # finite, infinite as bf16 (one a row: with two, whether a sum overflows is a matter of order)
    a[302, :] = 0.0
    a[302, 8] = 3.4e38
    b[8, 40:60] = 0.0
    b[100, 70] = np.inf
    b[101, 71] = np.nan
    a[400, :] *= np.float32(1e-38)          # parts below bf16's range without the scale
    a[401, :] *= np.float32(1e-42)          # subnormals
    a[402, :] *= np.float32(1e30)           # sums past the scaled range
    b[:, 90] *= np.float32(1e-20)
    got, path = product(vh, a, b, akc, bkc)
    assert path == vh.GEMM_PATH_PERSISTENT
    want, _ = product(vh, a, b, akc, bkc, engine=vh.GEMM_ENGINE_WIDE)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    np.testing.assert_array_equal(got[inf], want[inf])
    fine = np.isfinite(want)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    with np.errstate(all="ignore"):
        ref, mag = a64 @ b64, np.abs(a64) @ np.abs(b64)
    # Sums below the normal range round to 2^-149.
    bound = (K + 2) * 2.0 ** -24 * mag + K * 2.0 ** -149
    with np.errstate(all="ignore"):
        bad = np.argwhere(fine & ~(np.abs(got - ref) <= bound))
    assert not len(bad), [(i, j, got[i, j], want[i, j], ref[i, j], bound[i, j]) for i, j in bad[:5]]


def test_split_product_broadcast_operand(vh):
    """An operand repeated along k (stride 0) and a k tail: nothing read past K counts."""
    M, N, K = 300, 260, 1001
    r = np.random.default_rng(9)
    col = r.standard_normal(M).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    A, B, C = dev(vh, col), dev(vh, b), out(vh, (M, N))
    d = gemm_desc(vh, M, N, K, A.ptr, 1, 0, B.ptr, N, 1, C.ptr, N)
    vh.check(vh.lib.vh_gemm(ctypes.byref(d), None))
    assert vh.lib.vh_gemm_last_path() == vh.GEMM_PATH_PERSISTENT
    got = fetch(vh, C, (M, N))
    ref = col[:, None].astype(np.float64) * b.astype(np.float64).sum(0)
    bound = (K + 2) * 2.0 ** -24 * np.abs(col)[:, None] * np.abs(b).astype(np.float64).sum(0)
    assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("K,one_signed", [(768, False), (3072, False), (16384, False), (16384, True)])
def test_split_product_error_is_no_larger(vh, K, one_signed):
    """2-norm error against float64 beside the f32 instruction's (the WIDE engine):
    of the elements no larger (1.05 for the draw), of their sums over 512 rows and 768
    columns within 3 times (a bias that all elements share would make it 16 to 28)."""
    M, N = 512, 768
    r = np.random.default_rng(K)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    if one_signed:
        a, b = np.abs(a), np.abs(b)
    ref = a.astype(np.float64) @ b.astype(np.float64)

    def errors(engine):
        d = product(vh, a, b, True, True, engine=engine)[0] - ref
        return [np.linalg.norm(x) for x in (d, d.sum(0), d.sum(1))]
    split, f32 = errors(vh.GEMM_ENGINE_DEFAULT), errors(vh.GEMM_ENGINE_WIDE)
    print("split errors", K, one_signed, split, f32, flush=True)
    assert split[0] <= 1.05 * f32[0]
    assert split[1] <= 3 * f32[1] and split[2] <= 3 * f32[2]  # (no drift common to a row or a column)


# ------------------------------------------------ the tiled kernel (kernels/gemm.h) --

#   M, N, K, floats off alignment: K <= 8 on the f32 instruction, then edges of its 64 x
#   64 tiles and of its 32-wide k tiles, one and several of each (its 128 x 128 tiles:
#   test_gemm_kernels_gpu.py).
TILE_SIZES = [(64, 64, 1, 0), (65, 63, 8, 1), (63, 65, 9, 0), (1, 200, 33, 3), (200, 1, 31, 0), (129, 127, 95, 2),
              (64, 128, 32, 0), (700, 130, 65, 1), (255, 300, 2049, 1), (2048, 191, 100, 0)]


@pytest.mark.parametrize("size", TILE_SIZES, ids=str)
@pytest.mark.parametrize("akc,bkc", LAYOUTS)
def test_tiled_product_sizes(vh, akc, bkc, size):
    M, N, K, off = size
    print("tiled", size, akc, bkc, flush=True)
    r = np.random.default_rng(M + N + K)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    got, path = product(vh, a, b, akc, bkc, off)
    assert path in (vh.GEMM_PATH_TILED, vh.GEMM_PATH_SPLIT_K)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    u = 2.0 ** -24  # (the f32 bound; the split's own two u per product only past K = 8)
    bound = (K * u / (1 - K * u)) * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    assert np.all(np.abs(got - ref) <= bound)


def test_tiled_product_special_values(vh):
    M, N, K = 150, 140, 70
    r = np.random.default_rng(4)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    a[5, 17], a[6, 69], a[100, 0], a[101, 3] = np.inf, -np.inf, np.nan, 3.4e38
    a[102, :] = 0.0
    b[40, 70], b[41, 71] = np.inf, np.nan
    b[3, 70] = 0.0  # (row 101's term overflows in f32 and not in float64: none beside an infinity)
    a[120, :] *= np.float32(1e-42)
    got, _ = product(vh, a, b, True, False)
    with np.errstate(all="ignore"):
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        want = (a64 @ b64).astype(np.float32)  # one overflowing term a row: its sign is the sum's
        bound = (K + 2) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)) + K * 2.0 ** -149
        np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
        near = np.abs(want) > 3.39e38  # f32's edge: the sum may or may not round to infinity
        np.testing.assert_array_equal(got[np.isinf(want) & ~near], want[np.isinf(want) & ~near])
        fine = np.isfinite(want) & ~near
        assert np.all(np.isfinite(got[fine])) and np.all(np.abs(got - want)[fine] <= bound[fine] * 1.01)


@pytest.mark.parametrize("akc", [True, False])
def test_tiled_product_far_apart_rows(vh, akc):
    """A leading dimension past the buffer loads' 32-bit offsets: element by element."""
    M, K, N, ld = (3, 40, 70, (1 << 22) + 1) if akc else (40, 3, 70, (1 << 22) + 1)
    r = np.random.default_rng(6)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    big = np.zeros((3, ld), np.float32)
    big[:, :40] = a if akc else a.T
    A, B, C = dev(vh, big), dev(vh, b), out(vh, (M, N))
    d = gemm_desc(vh, M, N, K, A.ptr, ld if akc else 1, 1 if akc else ld, B.ptr, N, 1, C.ptr, N)
    vh.check(vh.lib.vh_gemm(ctypes.byref(d), None))
    ref = a.astype(np.float64) @ b.astype(np.float64)
    bound = (K + 2) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    assert np.all(np.abs(fetch(vh, C, (M, N)) - ref) <= bound)


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("K", [4, 8, 12, 32, 36, 64, 256])
def test_streamed_tiles(vh, akc, bkc, K, causal):
    """Batched short-K products as a stream of 128 x 128 tiles: edge tiles, one to
    eight k tiles and a ragged last one, K <= 8 on the f32 instruction, an infinity
    and a NaN in one batch (their own outputs alone), more tiles than workgroups."""
    nb, M, N = 140, 132, 260
    print("stream", akc, bkc, K, causal, flush=True)
    r = np.random.default_rng(K)
    a = r.standard_normal((nb, M, K)).astype(np.float32)
    b = r.standard_normal((nb, K, N)).astype(np.float32)
    a[77, 130, 2], a[77, 3, 1] = np.inf, np.nan
    A = dev(vh, np.ascontiguousarray(a if akc else np.swapaxes(a, 1, 2)))
    B = dev(vh, np.ascontiguousarray(np.swapaxes(b, 1, 2) if bkc else b))
    C = out(vh, (nb, M, N))
    d = gemm_desc(vh, M, N, K, A.ptr, K if akc else 1, 1 if akc else M, B.ptr, 1 if bkc else N, K if bkc else 1,
                  C.ptr, N, batch=(nb // 10, 10), a_sb=(10 * M * K, M * K), b_sb=(10 * K * N, K * N),
                  c_sb=(10 * M * N, M * N), causal=vh.GEMM_SKIP_UPPER if causal else 0)
    vh.check(vh.lib.vh_gemm(ctypes.byref(d), None))
    assert vh.lib.vh_gemm_last_path() == vh.GEMM_PATH_BATCHED
    got = fetch(vh, C, (nb, M, N))
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref, mag = a64 @ b64, np.abs(a64) @ np.abs(b64)
    u = 2.0 ** -24
    keep = np.tril(np.ones((M, N), bool)) if causal else np.ones((M, N), bool)  # (what causal = 1 defines)
    fine = np.isfinite(ref) & keep
    assert np.all(np.abs(got - ref)[fine] <= (K * u / (1 - K * u)) * mag[fine])
    odd = ~np.isfinite(ref) & keep
    np.testing.assert_array_equal(got[odd], ref[odd].astype(np.float32))
