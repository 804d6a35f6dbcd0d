"""Which kernel carries a product (vh_gemm_last_kernel), and what that choice must
not cost: the tests of the other files name a kernel's sizes, this one holds the
rule that picks it."""
import ctypes

import numpy as np
import pytest

from parity import dev, out
from test_block_ops_gpu import gemm_desc

pytestmark = pytest.mark.gpu


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
