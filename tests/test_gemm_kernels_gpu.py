"""Each product kernel at sizes that reach it, asserted by its name
(vh_gemm_last_kernel): edges, k tails, every form of the last round, epilogues, batches
and special values on the 256-row split kernel (kernels/gemm_split.h), the 128 x 128
tiles of kernels/gemm.h, the f32 kernel's narrow tile (kernels/gemm_big.h); and on all
of them, that an output does not depend on another row's or column's values.

Bound: as in test_gemm_split_gpu.py, (K + 2) u sum |a||b| with u = 2^-24."""
import ctypes
import functools

import numpy as np
import pytest

from parity import dev, fetch, out
from test_block_ops_gpu import gemm_desc

pytestmark = pytest.mark.gpu

LAYOUTS = [(True, True), (True, False), (False, True), (False, False)]


def product(vh, a, b, akc, bkc, off=0, ldx=0, pad=0.0, **kw):
    """vh_gemm of a [.., M, K] and b [.., K, N] stored k- or row-contiguous, `off` floats into
    their buffers, `ldx` further floats of value `pad` after each row; and its kernel."""
    nb, M, K = (1,) * (3 - a.ndim) + a.shape
    N = b.shape[-1]

    def put(x):
        x = x.reshape((nb,) + x.shape[-2:])
        x = np.pad(x, ((0, 0), (0, 0), (0, ldx)), constant_values=pad)
        return dev(vh, np.concatenate([np.zeros(off, np.float32), x.reshape(-1)])), x.shape[2], x.shape[1] * x.shape[2]
    A, lda, sa = put(a if akc else np.swapaxes(a, -1, -2))
    B, ldb, sb = put(np.swapaxes(b, -1, -2) if bkc else b)
    C = kw.pop("C", None) or out(vh, (nb, M, N))
    d = gemm_desc(vh, M, N, K, A.ptr + 4 * off, lda if akc else 1, 1 if akc else lda, B.ptr + 4 * off, 1 if bkc else ldb,
                  ldb if bkc else 1, C.ptr, N, batch=(1, nb), a_sb=(0, sa), b_sb=(0, sb), c_sb=(0, M * N), **kw)
    vh.check(vh.lib.vh_gemm(ctypes.byref(d), None))
    kernel = vh.lib.vh_gemm_last_kernel().decode()
    return fetch(vh, C, (nb, M, N)).reshape(a.shape[:-1] + (N,)), kernel


@functools.lru_cache(maxsize=1)
def operands(M, N, K, nb=0):
    r = np.random.default_rng(M + N + K)
    a = r.standard_normal(((nb,) if nb else ()) + (M, K)).astype(np.float32)
    b = r.standard_normal(((nb,) if nb else ()) + (K, N)).astype(np.float32)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    return a, b, a64 @ b64, np.abs(a64) @ np.abs(b64)


#   M, N, K, floats off 16-byte alignment, tile width
SPLIT_SIZES = [
    (4100, 2310, 701, 0, 192),   # rows and columns past a tile, k tail of 13, a round left whole, two chains
    (5003, 5001, 33, 1, 256),    # two k tiles and one k of a third, full round and a partly filled one
    (5000, 5000, 3, 0, 256),     # less than a k tile
    (600, 700, 9001, 3, 192),    # 12 tiles split over all workgroups, k tail of 9
    (770, 1000, 9001, 0, 256),   # the same, 256 wide
    (65600, 192, 400, 0, 192),   # 257 tiles: the last one's 25 k tiles leave most workgroups an empty run
]


@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("size", SPLIT_SIZES, ids=str)
def test_split_kernel_sizes(vh, size, akc, bkc):
    M, N, K, off, bn = size
    print("split", size, akc, bkc, flush=True)
    a, b, ref, mag = operands(M, N, K)
    got, kernel = product(vh, a, b, akc, bkc, off)
    assert kernel == f"vh_gemms_{'k' if akc else 'm'}{'k' if bkc else 'n'}_{bn}"
    assert np.all(np.abs(got - ref) <= (K + 2) * 2.0 ** -24 * mag)
    np.testing.assert_array_equal(product(vh, a, b, akc, bkc, off)[0], got)


@pytest.mark.parametrize("epi", ["bias", "full", "accumulate", "full accumulate alpha"])
@pytest.mark.parametrize("size", [(4100, 2310, 701, 0), (600, 700, 9001, 0), (300, 260, 9001, 4), (768, 768, 1024, 12)], ids=str)
def test_split_kernel_epilogues(vh, size, epi):
    """Whole tiles, edge tiles and pieces with every addend, over batches too."""
    M, N, K, nb = size
    print("split epilogue", size, epi, flush=True)
    a, b, ref, mag = operands(M, N, K, nb)
    r = np.random.default_rng(5)
    shape = ref.shape
    kw, want = {}, ref
    if "alpha" in epi:
        kw["alpha"] = 0.75
        want = 0.75 * want
    if "accumulate" not in epi or "full" in epi:
        e = r.standard_normal(shape if "full" in epi else (N,)).astype(np.float32)
        E = dev(vh, e)
        kw.update(e=E.ptr, e_sm=N if "full" in epi else 0, e_sn=1, e_sb=(0, M * N if "full" in epi else 0))
        want, mag = want + e, mag + np.abs(e)
    if "accumulate" in epi:
        c0 = r.standard_normal(shape).astype(np.float32)
        kw.update(accumulate=1, C=dev(vh, c0))
        want, mag = want + c0, mag + np.abs(c0)
    got, kernel = product(vh, a, b, True, False, **kw)
    assert kernel.startswith("vh_gemms_kn")
    assert np.all(np.abs(got - want) <= (K + 5) * 2.0 ** -24 * mag)


def test_split_kernel_broadcast_operand(vh):
    """An operand repeated along k (stride 0) and a k tail: nothing read past K counts."""
    M, N, K = 4100, 2310, 701
    r = np.random.default_rng(9)
    col = r.standard_normal(M).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    A, B, C = dev(vh, col), dev(vh, b), out(vh, (M, N))
    d = gemm_desc(vh, M, N, K, A.ptr, 1, 0, B.ptr, N, 1, C.ptr, N)
    vh.check(vh.lib.vh_gemm(ctypes.byref(d), None))
    assert vh.lib.vh_gemm_last_kernel().decode().startswith("vh_gemms_mn")
    got = fetch(vh, C, (M, N))
    ref = col[:, None].astype(np.float64) * b.astype(np.float64).sum(0)
    bound = (K + 2) * 2.0 ** -24 * np.abs(col)[:, None] * np.abs(b).astype(np.float64).sum(0)
    assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("M,N,K", [(4100, 2310, 701), (600, 700, 9001)])
def test_split_kernel_special_values(vh, M, N, K, akc, bkc):
    """Each special value where the f32 instruction (the WIDE engine) puts it, in whole
    tiles and in pieces; the other elements within the bound of their own exact sums."""
    print("split specials", M, N, K, akc, bkc, flush=True)
    a, b = (x.copy() for x in operands(M, N, K)[:2])
    a[5, 17] = np.inf
    a[6, K - 1] = -np.inf
    a[300, 0] = np.nan
    a[301, 3] = -3.4e38  # finite, infinite as bf16 (one a row: with two, whether a sum overflows is a matter of order)
    a[302, :] = 0.0
    a[302, 8] = 3.4e38
    b[8, 40:60] = 0.0
    b[100, 70] = np.inf
    b[101, N - 1] = np.nan
    a[400, :] *= np.float32(1e-38)          # parts below bf16's range without the scale
    a[401, :] *= np.float32(1e-42)          # subnormals
    a[402, :] *= np.float32(1e30)           # sums past the scaled range
    b[:, 90] *= np.float32(1e-20)
    got, kernel = product(vh, a, b, akc, bkc)
    assert kernel.startswith("vh_gemms")
    want, kernel = product(vh, a, b, akc, bkc, engine=vh.GEMM_ENGINE_WIDE)
    assert kernel.startswith("vh_gemmb")
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    np.testing.assert_array_equal(got[inf], want[inf])
    fine = np.isfinite(want)
    with np.errstate(all="ignore"):
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        ref, mag = a64 @ b64, np.abs(a64) @ np.abs(b64)
        # Sums below the normal range round to 2^-149.
        bad = np.argwhere(fine & ~(np.abs(got - ref) <= (K + 2) * 2.0 ** -24 * mag + K * 2.0 ** -149))
    assert not len(bad), [(i, j, got[i, j], want[i, j], ref[i, j]) for i, j in bad[:5]]


def test_split_kernel_empty_runs_after_workspace_reuse(vh):
    """With fewer k tiles in the last round than workgroups some write no piece: the fix-up
    must skip their slots, which hold what an earlier product left."""
    a, b, _, _ = operands(600, 700, 9001)
    assert product(vh, a, b, True, True)[1] == "vh_gemms_kk_192"  # 12 tiles: a piece from every workgroup
    M, N, K = 65600, 192, 400
    a, b, ref, mag = operands(M, N, K)
    got, kernel = product(vh, a, b, True, True)
    assert kernel == "vh_gemms_kk_192"
    assert np.all(np.abs(got - ref) <= (K + 2) * 2.0 ** -24 * mag)


@pytest.mark.parametrize("K,one_signed", [(768, False), (768, True), (3072, False), (3072, True)])
def test_split_kernel_error_is_no_larger(vh, K, one_signed):
    """Whole chains of K on both sides (256 tiles of 256 x 256: one round): 2-norm error
    against float64 beside the f32 instruction's, of the elements no larger (1.05 for the
    draw). Of their sums over rows and columns within 3 times (a bias that all elements
    share would make it 16 and more); of one-signed operands, whose small part products
    are lost under the sum alike along a row or column, within 2^-23 of the sum
    (a unit in its last place; measured 0.4)."""
    if vh.lib.vh_device_cu_count() // 8 * 8 != 256:
        pytest.skip("one full round needs 256 workgroups")
    a, b, ref, _ = operands(4096, 4096, K)
    if one_signed:
        a, b = np.abs(a), np.abs(b)
        ref = a.astype(np.float64) @ b.astype(np.float64)

    def errors(engine, name):
        got, kernel = product(vh, a, b, True, True, engine=engine)
        assert kernel == name
        d = got - ref
        return np.array([np.linalg.norm(x) for x in (d, d.sum(0), d.sum(1))])
    split = errors(vh.GEMM_ENGINE_DEFAULT, "vh_gemms_kk_256")
    f32 = errors(vh.GEMM_ENGINE_WIDE, "vh_gemmb_kk_256")
    print("split errors", K, one_signed, split, f32, flush=True)
    assert split[0] <= 1.05 * f32[0]
    if one_signed:
        assert np.all(split[1:] <= 2.0 ** -23 * np.array([np.linalg.norm(ref.sum(i)) for i in (0, 1)]))
    else:
        assert np.all(split[1:] <= 3 * f32[1:])


#   M, N, K, batches, engine, kernel
NEIGHBOURS = [
    (4100, 2310, 701, 0, 0, "vh_gemms"), (600, 700, 9001, 0, 0, "vh_gemms"),    # whole tiles; pieces
    (1000, 777, 1007, 0, 0, "vh_gemmt"), (500, 520, 32769, 0, 0, "vh_gemmt"),   # 64 x 64 and 128 x 128 tiles walked
    (200, 150, 100, 0, 0, "vh_gemm_"), (4097, 4100, 100, 0, 1, "vh_gemm_"),     # tiled, 64 and 128
    (132, 260, 64, 140, 0, "vh_gemmp"),
]


@pytest.mark.parametrize("akc,bkc", [(True, False), (False, True)])
@pytest.mark.parametrize("case", NEIGHBOURS, ids=str)
def test_outputs_do_not_depend_on_other_rows(vh, case, akc, bkc):
    """An infinity and a NaN in two rows and a column: every other output keeps its bits."""
    M, N, K, nb, engine, name = case
    print("neighbours", case, akc, bkc, flush=True)
    r = np.random.default_rng(8)
    a = r.standard_normal(((nb,) if nb else ()) + (M, K)).astype(np.float32)
    b = r.standard_normal(((nb,) if nb else ()) + (K, N)).astype(np.float32)
    clean, kernel = product(vh, a, b, akc, bkc, engine=engine)
    assert kernel.startswith(name), kernel
    a[..., 5, 17], a[..., 130, 3], b[..., 8, 60] = np.inf, np.nan, -np.inf
    got, _ = product(vh, a, b, akc, bkc, engine=engine)
    rows, cols = np.arange(M), np.arange(N)
    keep = np.ix_((rows != 5) & (rows != 130), cols != 60)
    assert np.all(np.isnan(got[..., 130, :])) and not np.any(np.isfinite(got[..., 5, :]))
    assert not np.any(np.isfinite(got[..., 60]))
    np.testing.assert_array_equal(got[(slice(None),) * (got.ndim - 2) + keep], clean[(slice(None),) * (got.ndim - 2) + keep])


@pytest.mark.parametrize("case", [c for c in NEIGHBOURS if c[3] == 0], ids=str)
def test_outputs_do_not_depend_on_padding(vh, case):
    """Infinities between the rows of row-contiguous operands, which edge tiles read."""
    M, N, K, nb, engine, name = case
    print("padding", case, flush=True)
    r = np.random.default_rng(8)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    zeros, kernel = product(vh, a, b, False, False, ldx=13, engine=engine)
    assert kernel.startswith(name), kernel
    infs, _ = product(vh, a, b, False, False, ldx=13, pad=np.inf, engine=engine)
    np.testing.assert_array_equal(infs, zeros)


# ---------------------------------------------------------- the tiled kernel's 128 x 128 tiles --

@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("M,N,K,off", [(4097, 4100, 100, 0), (5000, 4001, 33, 1), (4100, 4100, 8, 3)])
def test_tiled_128(vh, M, N, K, off, akc, bkc):
    """One pass over K on 128 x 128 tiles: edges, k tails, K <= 8 (the f32 instruction) and an
    infinity."""
    print("tiled 128", M, N, K, off, akc, bkc, flush=True)
    a, b = (x.copy() for x in operands(M, N, K)[:2])
    a[200, 1], b[2, 300] = np.inf, -np.inf
    got, kernel = product(vh, a, b, akc, bkc, off, engine=vh.GEMM_ENGINE_TILED)
    assert kernel == f"vh_gemm_{'k' if akc else 'm'}4_{'k' if bkc else 'n'}4"
    with np.errstate(invalid="ignore"):
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        ref, mag = a64 @ b64, np.abs(a64) @ np.abs(b64)
    odd = ~np.isfinite(ref)
    np.testing.assert_array_equal(got[odd], ref[odd].astype(np.float32))
    assert np.all(np.abs(got[~odd] - ref[~odd]) <= K * 2.0 ** -24 / (1 - K * 2.0 ** -24) * mag[~odd])


# ------------------------------------------------ the f32 kernel's 256 x 192 tile --

@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("M,N,K", [(512, 192, 1024), (777, 255, 2050), (300, 200, 16384)])
def test_f32_kernel_narrow_tile(vh, M, N, K, akc, bkc):
    """192 to 255 columns under the WIDE engine, the split round and a k tail."""
    print("f32 narrow", M, N, K, akc, bkc, flush=True)
    a, b, ref, mag = operands(M, N, K)
    got, kernel = product(vh, a, b, akc, bkc, engine=vh.GEMM_ENGINE_WIDE)
    assert kernel == f"vh_gemmb_{'k' if akc else 'm'}{'k' if bkc else 'n'}_192"
    assert np.all(np.abs(got - ref) <= K * 2.0 ** -24 / (1 - K * 2.0 ** -24) * mag)
    np.testing.assert_array_equal(product(vh, a, b, akc, bkc, engine=vh.GEMM_ENGINE_WIDE)[0], got)
