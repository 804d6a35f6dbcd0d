"""Which kernel carries a product (vh_gemm_last_kernel), and what that choice must
not cost: the tests of the other files name a kernel's sizes, this one holds the
rule that picks it."""
import ctypes

import numpy as np
import pytest

from parity import dev, fetch, out
from test_block_ops_gpu import gemm_desc

pytestmark = pytest.mark.gpu


def product(vh, a, b, akc, bkc, **kw):
    """vh_gemm of a [M, K] and b [K, N] stored k- or row-contiguous, and its kernel."""
    M, K = a.shape
    N = b.shape[1]
    A, B = dev(vh, np.ascontiguousarray(a if akc else a.T)), dev(vh, np.ascontiguousarray(b.T if bkc else b))
    C = out(vh, (M, N))
    d = gemm_desc(vh, M, N, K, A.ptr, K if akc else 1, 1 if akc else M, B.ptr, 1 if bkc else N, K if bkc else 1, C.ptr,
                  N, **kw)
    vh.check(vh.lib.vh_gemm(ctypes.byref(d), None))
    kernel = vh.lib.vh_gemm_last_kernel().decode()
    return fetch(vh, C, (M, N)), kernel


def test_last_kernel_names_the_product_kernel(vh):
    X, C = dev(vh, np.zeros(1 << 21, np.float32)), out(vh, (1 << 20,))

    def kernel(M, N, K, **kw):
        d = gemm_desc(vh, M, N, K, X.ptr, K, 1, X.ptr, 1, K, C.ptr, N, **kw)
        vh.check(vh.lib.vh_gemm(ctypes.byref(d), None))
        return vh.lib.vh_gemm_last_kernel().decode()
    assert kernel(1024, 1000, 1000) == "vh_gemmt_kk"
    assert kernel(512, 512, 2048, engine=vh.GEMM_ENGINE_WIDE) == "vh_gemmb_kk_256"
    assert kernel(512, 192, 2050, engine=vh.GEMM_ENGINE_WIDE) == "vh_gemmb_kk_192"  # not its k tail's
    assert kernel(70, 50, 30) == "vh_gemm_k4_k4_t64"
    assert kernel(0, 50, 30) == ""


@pytest.mark.parametrize("akc,bkc", [(True, True), (False, False)])
@pytest.mark.parametrize("M,N,K", [(8192, 8192, 1), (6000, 6000, 2), (5000, 5000, 3), (3000, 3000, 8)])
def test_few_k_error(vh, M, N, K, akc, bkc):
    """The bound of a chain of K f32 multiply-adds (u = 2^-24), which a split product, up
    to 1.9 u off, does not meet below K = 3; at K = 1 the f32 product itself."""
    print("few k", M, N, K, akc, bkc, flush=True)
    r = np.random.default_rng(K)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    got, kernel = product(vh, a, b, akc, bkc)
    assert kernel.startswith("vh_gemms") == (K > 2), kernel
    if K == 1:
        np.testing.assert_array_equal(got, a * b)
    a64, b64, u = a.astype(np.float64), b.astype(np.float64), 2.0 ** -24
    assert np.all(np.abs(got - a64 @ b64) <= K * u / (1 - K * u) * (np.abs(a64) @ np.abs(b64)))
