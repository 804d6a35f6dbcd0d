"""Each product kernel at sizes that reach it, asserted by its name
(vh_gemm_last_kernel): an output does not depend on another row's or column's values."""
import ctypes

import numpy as np
import pytest

from parity import dev, fetch, out
from test_block_ops_gpu import gemm_desc

pytestmark = pytest.mark.gpu


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
