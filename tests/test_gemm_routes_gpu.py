"""Which kernel carries a product (vh_gemm_last_kernel), and what that choice must
not cost: the tests of the other files name a kernel's sizes, this one holds the
rule that picks it."""
import ctypes
import fnmatch

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


def f32_chain(a, b):
    """a b as one chain of f32 fused multiply-adds in k order (float64 holds a product exactly)."""
    s = np.zeros((a.shape[0], b.shape[1]), np.float32)
    for k in range(a.shape[1]):
        s = (s + a[:, k:k + 1].astype(np.float64) * b[k]).astype(np.float32)
    return s


#   M, N, K with 256 x 192 tiles short of one round of workgroups: edges, several k
#   lengths, two and three chains, and a k tile too few for more
SHORT_ROUNDS = [(10000, 768, 384), (14000, 500, 200), (2048, 4096, 768), (3000, 2304, 512), (11000, 770, 515),
                (15000, 700, 900)]


@pytest.mark.parametrize("akc,bkc", [(True, True), (False, False)])
@pytest.mark.parametrize("M,N,K", SHORT_ROUNDS)
def test_short_round_error(vh, M, N, K, akc, bkc):
    """t tiles short of a round of G workgroups: no less exact than f32 sums in the pieces
    that a round split over all workgroups has (cut every t K / G of the tiles' joined k
    ranges). Such a chain of l out of K terms has (l / K)^2 of the whole chain's error
    variance, which grows with the square of the length."""
    print("short round", M, N, K, akc, bkc, flush=True)
    r = np.random.default_rng(M + K)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    got, kernel = product(vh, a, b, akc, bkc)
    G, t = vh.lib.vh_device_cu_count() // 8 * 8, -(-M // 256) * -(-N // 192)
    assert kernel.startswith("vh_gemms") and t < G
    cuts = np.union1d(np.arange(t + 1) * G, np.arange(G + 1) * t) / (t * G)  # of the joined range, in [0, 1]
    pieces = np.sqrt(np.sum((np.diff(cuts) * t) ** 2) / t)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    rows = slice(0, 200)
    f32 = np.linalg.norm(f32_chain(a[rows], b) - ref[rows])
    split = np.linalg.norm(got[rows] - ref[rows])
    print("error / the pieces'", split / (f32 * pieces), flush=True)
    assert split <= 1.05 * f32 * pieces
    bound = (K + 2) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64))
    assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("epi", ["bias", "full", "accumulate", "full accumulate alpha", "batch"])
def test_chains_epilogue(vh, epi):
    """A tile summed in two chains applies the addend and the old C once, alpha to both."""
    print("chains", epi, flush=True)
    nb, M, N, K = (2, 4500, 770, 768) if epi == "batch" else (1, 9001, 770, 768)
    r = np.random.default_rng(4)
    a = r.standard_normal((nb, M, K)).astype(np.float32)
    b = r.standard_normal((nb, K, N)).astype(np.float32)
    c0 = r.standard_normal((nb, M, N)).astype(np.float32)
    e = r.standard_normal((nb, M, N) if "full" in epi or epi == "batch" else (N,)).astype(np.float32)
    A, B, C, E = dev(vh, a), dev(vh, b), dev(vh, c0), dev(vh, e)
    kw = {}
    want = a.astype(np.float64) @ b.astype(np.float64)
    mag = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    if "alpha" in epi:
        kw["alpha"] = 0.75
        want *= 0.75
    if epi != "accumulate":
        kw.update(e=E.ptr, e_sm=N if e.ndim == 3 else 0, e_sn=1, e_sb=(0, M * N) if e.ndim == 3 else (0, 0))
        want, mag = want + e, mag + np.abs(e)
    if "accumulate" in epi:
        kw["accumulate"] = 1
        want, mag = want + c0, mag + np.abs(c0)
    d = gemm_desc(vh, M, N, K, A.ptr, K, 1, B.ptr, N, 1, C.ptr, N, batch=(1, nb), a_sb=(0, M * K), b_sb=(0, K * N),
                  c_sb=(0, M * N), **kw)
    vh.check(vh.lib.vh_gemm(ctypes.byref(d), None))
    assert vh.lib.vh_gemm_last_kernel().decode().startswith("vh_gemms")
    got = fetch(vh, C, (nb, M, N))
    assert np.all(np.abs(got - want) <= (K + 5) * 2.0 ** -24 * mag)


@pytest.mark.parametrize("akc,bkc", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("M,N,K,want", [(256, 256, 65536, "vh_gemmt_??"), (300, 500, 16385, "vh_gemmt_??"),
                                        (500, 520, 32769, "vh_gemmt_??_128"), (512, 768, 50272, "vh_gemmt_??_128"),
                                        (2000, 1500, 17000, "vh_gemms_??_*")])
def test_few_outputs_of_long_k(vh, M, N, K, want, akc, bkc):
    """Few outputs over a K past 16384 walk the smaller tiles' K ranges in one launch;
    more run on the 256-row tiles, a launch per range of K. The f32 instruction's error
    bounds both, of the elements and of their sums over rows and columns (3: a drift
    common to all would be 10 and more)."""
    print("long k", M, N, K, akc, bkc, flush=True)
    r = np.random.default_rng(K)
    a = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    got, kernel = product(vh, a, b, akc, bkc)
    assert fnmatch.fnmatch(kernel, want), kernel
    f32 = product(vh, a, b, akc, bkc, engine=vh.GEMM_ENGINE_WIDE)[0]
    ref = a.astype(np.float64) @ b.astype(np.float64)
    d, e = got - ref, f32 - ref
    assert np.linalg.norm(d) <= 1.05 * np.linalg.norm(e)
    assert np.linalg.norm(d.sum(0)) <= 3 * np.linalg.norm(e.sum(0))
    assert np.linalg.norm(d.sum(1)) <= 3 * np.linalg.norm(e.sum(1))
