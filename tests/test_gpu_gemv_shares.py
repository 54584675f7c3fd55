"""The matrix-vector kernel (mmt4d_gemv.hip) where its four wavefronts' shares of K are empty, shorter than the ring of eight
loads, one ring, one and some, two; with and without a K that ends inside a step; and on both sides of the lines at which a
rhs tile is dealt to one, two or four workgroups (3/16, 1/2, 1 and 3/2 of 256 compute units; at most 4 and 8 lhs rows), with
lhs rows in one tile and in several, strided and accumulating.

Integers are compared bit for bit with a float64 product, floats within 1e-3 of max(|ref|, rms(ref)): sums of at most
67600 products of unit-scale values in 32 bits differ by about 1e-6 of that in any order.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

S8, F16, BF16 = abi.MMT4D_TYPE_S8S8S32, abi.MMT4D_TYPE_F16F16F32, abi.MMT4D_TYPE_BF16BF16F32
STEPS = [1, 3, 4, 5, 31, 32, 33, 60, 64, 65, 100]  # of 64 bytes of K; a split tile takes 2 or 4 of them at once


@pytest.mark.parametrize("flags,K0", [(BF16, 8), (F16, 16), (S8, 64), (S8, 16), (S8, 32)])
@pytest.mark.parametrize("M,M0", [(1, 1), (3, 1), (1, 4), (5, 1), (1, 8), (2, 4), (9, 1), (1, 16)])
def test_shares(gpu_lib, flags, K0, M, M0):  # noqa: F811
    e = 1 if flags == S8 else 2
    tiles = [16, 48, 49, 128, 129, 255, 257, 384, 385] if M * M0 <= 8 else [16, 255, 257]
    for n, steps in enumerate(STEPS):
        N = tiles[(n + M) % len(tiles)]
        for K in {steps * 64 // (K0 * e), steps * 64 // (K0 * e) + (1 if K0 * e < 64 else 0)}:
            pad = 16 // e if n % 2 else 0
            run_case(gpu_lib, flags, M, N, K, M0, 16, K0, "mmt4d_gemv*", lhs_pad=pad, rhs_pad=2 * pad,
                     out_pad=4 if n % 2 else 0, offsets=(pad, 2 * pad, 4 if n % 2 else 0), accumulate=n % 3 == 1, seed=n)
    for N in tiles:
        run_case(gpu_lib, flags, M, N, 2304 // (K0 * e) + 1, M0, 16, K0, "mmt4d_gemv", seed=N)


@pytest.mark.parametrize("K0", [32, 64])
@pytest.mark.parametrize("M,M0", [(1, 1), (7, 1), (2, 4), (9, 1), (1, 16)])
def test_int4_shares(gpu_lib, K0, M, M0):  # noqa: F811
    # (a step is 128 values; the ring is 4, 6 or 8 steps long; 1030 tiles of 58 KB and more come from HBM)
    for n, values in enumerate([128, 160, 192, 256, 480, 1920, 2048, 2080, 2112, 3072, 3104, 4000, 4128, 6336, 12000]):
        for N in {[16, 128, 129, 255, 257, 384, 385][(n + M) % 7], 771 + n if values < 4000 else 31}:
            pad = 32 if n % 2 else 0
            run_case(gpu_lib, abi.MMT4D_TYPE_S8S4S32, M, N, values // K0, M0, 16, K0, "mmt4d_gemv*", lhs_pad=pad,
                     rhs_pad=2 * pad, out_pad=4 if n % 2 else 0, offsets=(pad, 2 * pad, 4 if n % 2 else 0),
                     accumulate=n % 3 == 1, seed=n)
    for N in (770, 1025, 1030):
        run_case(gpu_lib, abi.MMT4D_TYPE_S8S4S32, M, N, 8320 // K0, M0, 16, K0, "mmt4d_gemv", seed=N)


# Few tiles dealt to two or four workgroups whose rhs is more than 48 MiB and read past the caches.
@pytest.mark.parametrize("flags,K0", [(BF16, 8), (F16, 16), (S8, 64), (S8, 16)])
@pytest.mark.parametrize("M,M0,N,row_bytes", [(1, 1, 320, 10304), (1, 8, 384, 8720), (1, 4, 300, 11000), (1, 1, 48, 66000), (3, 1, 47, 67584),
                                              (1, 8, 128, 25104)])
def test_split_tiles_from_hbm(gpu_lib, flags, K0, M, M0, N, row_bytes):  # noqa: F811
    K = row_bytes // (K0 * (1 if flags == S8 else 2))
    run_case(gpu_lib, flags, M, N, K, M0, 16, K0, "mmt4d_gemv", accumulate=M == 3, seed=N)


@pytest.mark.parametrize("K0", [32, 64])
@pytest.mark.parametrize("M,M0,N,depth", [(1, 1, 384, 16512), (1, 8, 300, 21216), (5, 1, 128, 49984)])
def test_int4_split_tiles_from_hbm(gpu_lib, K0, M, M0, N, depth):  # noqa: F811
    run_case(gpu_lib, abi.MMT4D_TYPE_S8S4S32, M, N, depth // K0, M0, 16, K0, "mmt4d_gemv", accumulate=M == 5, seed=N)
