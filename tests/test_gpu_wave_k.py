"""The mmt4d kernel that splits K over the wavefronts of a workgroup (mmt4d_wave_k_kernels.h): every type, row piece size
and output type it is instantiated for, on every tile that the host takes for them (16 to 64 rows and columns), at sizes
that the tiles do not divide, with K from less than a batch of steps per wavefront to many, ending on a step and inside one,
strided and accumulating; and with weights that are read past the caches.

Integers are compared bit for bit with a float64 product, floats within 1e-3 of max(|ref|, rms(ref)): sums of at most
5000 products of unit-scale values in 32 bits differ by about 1e-6 of that in any order, 16-bit results by one unit in
their last place besides.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

LAYOUTS = [
    (abi.MMT4D_TYPE_S8S8S32, 16, 16, 64), (abi.MMT4D_TYPE_S8S8S32, 8, 8, 4), (abi.MMT4D_TYPE_S8S8S32, 16, 16, 2),
    (abi.MMT4D_TYPE_S8S8S32, 8, 16, 2), (abi.MMT4D_TYPE_S8S8S32, 2, 16, 8), (abi.MMT4D_TYPE_S8S8S32, 1, 16, 32),
    (abi.MMT4D_TYPE_F16F16F32, 16, 16, 16), (abi.MMT4D_TYPE_F16F16F32, 16, 16, 1), (abi.MMT4D_TYPE_F16F16F32, 8, 8, 1),
    (abi.MMT4D_TYPE_BF16BF16F32, 8, 8, 4), (abi.MMT4D_TYPE_BF16BF16F32, 4, 16, 2), (abi.MMT4D_TYPE_BF16BF16F32, 1, 4, 16),
    (abi.MMT4D_TYPE_F32F32F32, 16, 16, 4), (abi.MMT4D_TYPE_F32F32F32, 16, 16, 1), (abi.MMT4D_TYPE_F32F32F32, 4, 8, 2),
    (abi.MMT4D_TYPE_F16F16F16, 16, 16, 16), (abi.MMT4D_TYPE_F16F16F16, 16, 16, 1), (abi.MMT4D_TYPE_BF16BF16BF16, 16, 16, 2),
    (abi.MMT4D_TYPE_BF16BF16BF16, 8, 8, 4), (abi.MMT4D_TYPE_S8S4S32, 16, 16, 32), (abi.MMT4D_TYPE_S8S4S32, 4, 16, 64),
]


@pytest.mark.parametrize("flags,M0,N0,K0", LAYOUTS)
def test_edges_of_tiles_and_of_K(gpu_lib, flags, M0, N0, K0):  # noqa: F811
    e = {abi.MMT4D_TYPE_S8S8S32: 1, abi.MMT4D_TYPE_S8S4S32: 1, abi.MMT4D_TYPE_F32F32F32: 4}.get(flags, 2)
    row_piece = K0 * e
    i4 = flags == abi.MMT4D_TYPE_S8S4S32
    for n, (rows, cols, row_bytes) in enumerate([(16, 16, 64), (20, 4000, 1100), (17, 40, 5000), (48, 1000, 2000),
                                                 (70, 264, 4500), (200, 520, 800), (1000, 1000, 1400)]):
        K = -(-row_bytes // row_piece)
        if i4 and K0 == 32:
            K |= 1
        elif not i4 and K * row_piece % 256 == 0:
            K += 1
        pad = 32 // e if n % 2 else 0
        run_case(gpu_lib, flags, -(-rows // M0), -(-cols // N0), K, M0, N0, K0,
                 "mmt4d_mfma_wave_k_*" if 0 < n < 6 else "mmt4d_mfma_*", lhs_pad=pad, rhs_pad=pad,
                 out_pad=4 if n % 2 else 0, offsets=(pad, pad, 4 if n % 2 else 0), accumulate=n % 3 == 1, seed=n)


# Sizes around where the host goes from one tile to the next, K short and long, ending inside a step of some wavefront's
# first batch and later: all tiles that the host takes for a layout are among what runs. 64x64 is not taken for f32 (bound
# by the matrix pipe) and hardly for row pieces of 4 and 8 bytes.
SIZES = [(20, 24, 300), (24, 72, 5000), (20, 3000, 300), (40, 1500, 5000), (40, 3000, 300), (100, 1500, 5000), (40, 6000, 600),
         (72, 5000, 5000), (200, 2500, 3000), (330, 1500, 4500), (264, 2000, 5000), (460, 1900, 1100)]


@pytest.mark.parametrize("flags,M0,N0,K0", LAYOUTS)
def test_every_tile(gpu_lib, flags, M0, N0, K0):  # noqa: F811
    e = {abi.MMT4D_TYPE_S8S8S32: 1, abi.MMT4D_TYPE_S8S4S32: 1, abi.MMT4D_TYPE_F32F32F32: 4}.get(flags, 2)
    seen = set()
    for n, (rows, cols, row_bytes) in enumerate(SIZES):
        K = -(-row_bytes // (K0 * e))
        if flags == abi.MMT4D_TYPE_S8S4S32 and K0 == 32:
            K |= 1  # half a step
        pad = 32 // e if n % 2 else 0
        run_case(gpu_lib, flags, -(-rows // M0), -(-cols // N0), K, M0, N0, K0, "mmt4d_mfma_*", lhs_pad=pad, rhs_pad=pad,
                 out_pad=4 if n % 2 else 0, offsets=(pad, pad, 4 if n % 2 else 0), accumulate=n % 3 == 0, seed=n)
        seen.add(gpu_lib.iree_uk_mi355x_last_kernel().decode())
    tiles = ["16x16", "16x32", "32x32", "32x64"] + ["64x64"] * (flags != abi.MMT4D_TYPE_F32F32F32 and not 4 <= K0 * e < 16)
    assert {"mmt4d_mfma_wave_k_" + t for t in tiles} <= seen, seen


# At most 256 tiles of 64x32, one for a compute unit, where there are more than 256 of 32x64.
@pytest.mark.parametrize("flags,M0,N0,K0", LAYOUTS)
def test_tiles_of_64x32_fill_the_units_once(gpu_lib, flags, M0, N0, K0):  # noqa: F811
    e = {abi.MMT4D_TYPE_S8S8S32: 1, abi.MMT4D_TYPE_S8S4S32: 1, abi.MMT4D_TYPE_F32F32F32: 4}.get(flags, 2)
    for n, (rows, cols, row_bytes) in enumerate([(190, 2700, 600), (304, 1620, 2100), (614, 790, 4300)]):
        K = -(-row_bytes // (K0 * e))
        if flags == abi.MMT4D_TYPE_S8S4S32 and K0 == 32:
            K |= 1
        pad = 32 // e if n % 2 else 0
        run_case(gpu_lib, flags, -(-rows // M0), -(-cols // N0), K, M0, N0, K0, "mmt4d_mfma_wave_k_64x32", lhs_pad=pad,
                 rhs_pad=pad, out_pad=4 if n % 2 else 0, offsets=(pad, pad, 4 if n % 2 else 0), accumulate=n % 3 == 0, seed=n)


# One row of tiles and more than 48 MiB of weights (row pieces of 16 bytes and more): non-temporal loads.
@pytest.mark.parametrize("flags,M0,N0,K0", [l for l in LAYOUTS if l[3] * {abi.MMT4D_TYPE_F32F32F32: 4}.get(l[0], 1) >= 16])
def test_weights_from_hbm(gpu_lib, flags, M0, N0, K0):  # noqa: F811
    i4 = flags == abi.MMT4D_TYPE_S8S4S32
    e = {abi.MMT4D_TYPE_S8S8S32: 1, abi.MMT4D_TYPE_S8S4S32: 1, abi.MMT4D_TYPE_F32F32F32: 4}.get(flags, 2)
    sizes = [(24, 28000, 4200), (48, 13000, 8300)] if i4 else [(24, 7000, 8000), (24, 13000, 4200), (48, 6500, 8300)]
    for n, (rows, cols, row_bytes) in enumerate(sizes):
        K = -(-row_bytes // (K0 * e)) | 1
        run_case(gpu_lib, flags, -(-rows // M0), -(-cols // N0), K, M0, N0, K0, "mmt4d_mfma_wave_k_*", accumulate=n == 0, seed=n)
