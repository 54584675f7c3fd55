"""The end of K on the block tiles (mmt4d_mfma_kernels.h): one chunk of 64 bytes per row, two, three, and K that ends inside
the second, the third or a later one: the first chunk then shares bytes with the second and is masked in front of the loop. Every
block tile, sizes that no tile divides, strided and accumulating.

Integers are compared bit for bit with a float64 product, floats within 1e-3 of max(|ref|, rms(ref)): sums of at most
1100 products of unit-scale values in 32 bits differ by about 1e-6 of that in any order.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

S8, S8S4, F16, BF16 = abi.MMT4D_TYPE_S8S8S32, abi.MMT4D_TYPE_S8S4S32, abi.MMT4D_TYPE_F16F16F32, abi.MMT4D_TYPE_BF16BF16F32
SMALL = {"64x64": (990, 696), "128x64": (1384, 968), "128x128": (680, 4504)}
LARGER = {tile: SMALL[tile] for tile in ("128x64", "128x128")}  # (the others take another kernel at 64x64's size)


@pytest.mark.parametrize("flags,T0,K0,tiles", [
    (S8S4, 16, 32, {"64x128": (1384, 968), "128x128": (680, 4504), "192x128": (2990, 2990), "256x128": (1980, 2970), "256x256": (4080, 4070)}),
    (BF16, 16, 16, LARGER), (S8, 8, 4, SMALL), (S8, 8, 8, LARGER), (F16, 16, 1, LARGER),
    (BF16, 16, 16, {"192x192": (2990, 2990), "256x192": (1350, 6990)})])
def test_chunks(gpu_lib, flags, T0, K0, tiles):  # noqa: F811
    e = 1 if flags in (S8, S8S4) else 2
    for tile, (rows, cols) in tiles.items():
        for n, row_bytes in enumerate([64, 96, 128, 160, 192, 2080]):
            pad = 32 // e if n % 2 else 0
            run_case(gpu_lib, flags, -(-rows // T0), -(-cols // T0), row_bytes // (K0 * e), T0, T0, K0,
                     "mmt4d_mfma_" + tile if n < 5 else "mmt4d_mfma_*", lhs_pad=pad, rhs_pad=2 * pad,
                     out_pad=4 if n % 2 else 0, offsets=(pad, 2 * pad, 4 if n % 2 else 0), accumulate=n % 3 == 1, seed=n)
