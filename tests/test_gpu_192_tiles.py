"""The block tiles with a side of 192 rows (mmt4d_mfma_kernels.h): every row piece size and type that has them, at sizes
that they do not divide and that the choice of tile gives to them, with K from one chunk of 64 bytes to several and ending
inside one, strided and accumulating.

Integers are compared bit for bit with a float64 product, floats within 1e-3 of max(|ref|, rms(ref)): sums of at most
3100 products of unit-scale values in 32 bits differ by about 1e-6 of that in any order, 16-bit results by one unit in
their last place besides.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

S8, S8S4, F16, BF16 = abi.MMT4D_TYPE_S8S8S32, abi.MMT4D_TYPE_S8S4S32, abi.MMT4D_TYPE_F16F16F32, abi.MMT4D_TYPE_BF16BF16F32
TALL = {"192x192": (2000, 4168), "128x192": (504, 11000), "192x128": (11000, 504), "256x192": (2808, 7832), "192x256": (568, 20472)}
SHAPES = {"pieces of 4 bytes and more": ["192x192", "128x192", "192x128", "256x192", "192x256"],
          "pieces of 2 bytes": ["256x192", "192x256"], "int4": ["192x128"]}


@pytest.mark.parametrize("flags,M0,N0,K0,have", [
    (S8, 8, 8, 4, 0), (S8, 16, 16, 64, 0), (S8, 8, 8, 8, 0), (S8, 1, 16, 64, 0), (S8, 16, 16, 2, 1), (S8, 8, 8, 2, 1),
    (F16, 16, 16, 16, 0), (F16, 16, 16, 1, 1), (BF16, 16, 16, 8, 0), (BF16, 16, 16, 2, 0), (BF16, 8, 8, 4, 0),
    (abi.MMT4D_TYPE_F16F16F16, 16, 16, 16, 0), (abi.MMT4D_TYPE_BF16BF16BF16, 16, 16, 2, 0),
    (abi.MMT4D_TYPE_F16F16F16, 16, 16, 1, 1), (S8S4, 16, 16, 32, 2)])
def test_ragged(gpu_lib, flags, M0, N0, K0, have):  # noqa: F811
    e = {S8: 1, S8S4: 1}.get(flags, 2)
    for n, tile in enumerate(list(SHAPES.values())[have]):
        rows, cols = TALL[tile]
        whole = 64 // (K0 * e) if K0 * e < 64 else 1  # k steps of a chunk
        # one chunk; a chunk and a bit (not with an int4 rhs, which takes whole chunks); several
        for K in {whole, whole + (whole if have == 2 else max(1, whole // 3)), 4 * whole}:
            pad = 32 // e if K % 2 else 0
            run_case(gpu_lib, flags, rows // M0, cols // N0, K, M0, N0, K0, "mmt4d_mfma_" + tile, lhs_pad=pad, rhs_pad=2 * pad,
                     out_pad=4 if n % 2 else 0, offsets=(pad, 2 * pad, 4 if n % 2 else 0), accumulate=K == 4 * whole, seed=n)


@pytest.mark.parametrize("flags,M0,N0,K0", [(S8, 8, 8, 4), (BF16, 16, 16, 16), (F16, 16, 16, 1), (abi.MMT4D_TYPE_BF16BF16BF16, 16, 16, 2)])
def test_deep_ring(gpu_lib, flags, M0, N0, K0):  # noqa: F811
    # Operands of more than 48 MiB on at most 256 tiles of 128x128: a ring of ten stages. K ends inside a chunk.
    e = 1 if flags == S8 else 2
    cols, row_bytes = 14300 // N0, 6000
    run_case(gpu_lib, flags, 152 // M0, cols, row_bytes // (K0 * e) + 1, M0, N0, K0, "mmt4d_mfma_128x128", accumulate=True, out_pad=4)
