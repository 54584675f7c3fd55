"""The kernel that splits K over wavefronts (mmt4d_wave_k_kernels.h): every tile that f32 has, in row pieces of 16 and 4 bytes
(loaded one at a time) and of 8 (staged), at sizes that the tile does not divide; and the 4-byte row pieces of the other types
on both sides of where they are loaded one at a time. K ends on a step and inside one, what lies behind it is NaN.

Integers are compared bit for bit with a float64 product, floats within 1e-3 of max(|ref|, rms(ref)): sums of at most
6000 products of unit-scale values in 32 bits differ by about 1e-6 of that in any order.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

TILES = {"16x16": (21, 59, 17), "16x32": (19, 2155, 17), "32x32": (33, 2946, 17), "32x48": (66, 2798, 17), "48x32": (176, 2027, 66),
         "32x64": (98, 3163, 66), "64x32": (174, 2700, 66), "48x48": (161, 2762, 131), "32x80": (193, 2462, 260),
         "80x32": (609, 962, 260), "48x64": (677, 903, 515), "64x48": (482, 1503, 515), "48x80": (257, 3309, 17),
         "80x48": (77, 11300, 260), "64x64": (250, 3970, 2050), "64x80": (291, 3420, 131), "80x64": (513, 2258, 131)}


# (64x64: staged, the block tile of that size is the faster one.)
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M0,N0,K0", [(16, 16, 4), (16, 16, 1), (8, 8, 1), (4, 8, 2)])
def test_f32(gpu_lib, M0, N0, K0, tile):  # noqa: F811
    rows, cols, depth = TILES[tile]
    for n, k in enumerate((depth, -(-depth // 16) * 16)):
        run_case(gpu_lib, abi.MMT4D_TYPE_F32F32F32, -(-rows // M0), -(-cols // N0), -(-k // K0), M0, N0, K0,
                 "mmt4d_mfma_*64x64" if tile == "64x64" else "mmt4d_mfma_wave_k_" + tile, lhs_pad=8 * n, rhs_pad=16 * n, out_pad=4 * n, offsets=(4 * n, 8 * n, 4 * n),
                 accumulate=n == 1, seed=n)


# One fragment, K on both sides of where two steps are in flight instead of one (32 steps of 16 values, K's end included).
@pytest.mark.parametrize("K0", [4, 1, 2])
def test_f32_long_K(gpu_lib, K0):  # noqa: F811
    for n, depth in enumerate((480, 495, 497, 512, 530, 1920, 5998)):
        run_case(gpu_lib, abi.MMT4D_TYPE_F32F32F32, 3, 5, -(-depth // K0), 16, 16, K0, "mmt4d_mfma_wave_k_16x16", accumulate=n % 2 == 1, seed=n)


# Rows, columns and bytes of K, and the tile they take: K that leaves the rows of 4-row operand tiles no round number of bytes
# apart, and K that leaves them a multiple of 512 apart (staged, test_mmt4d_choice_on_host.py).
FOUR_BYTE_LAYOUTS = [
    (abi.MMT4D_TYPE_S8S8S32, 16, 16, 4), (abi.MMT4D_TYPE_S8S8S32, 8, 8, 4), (abi.MMT4D_TYPE_S8S8S32, 4, 16, 4),
    (abi.MMT4D_TYPE_S8S8S32, 4, 8, 4), (abi.MMT4D_TYPE_S8S8S32, 8, 4, 4),
    (abi.MMT4D_TYPE_BF16BF16F32, 16, 16, 2), (abi.MMT4D_TYPE_BF16BF16F32, 8, 16, 2), (abi.MMT4D_TYPE_BF16BF16F32, 8, 8, 2),
    (abi.MMT4D_TYPE_BF16BF16F32, 4, 16, 2), (abi.MMT4D_TYPE_F16F16F32, 16, 8, 2), (abi.MMT4D_TYPE_F16F16F16, 16, 16, 2)]
FOUR_BYTE_SIZES = [(20, 24, 2100, "16x16"), (20, 3000, 700, "16x32"), (100, 1500, 2700, "32x32"), (100, 3000, 1600, "32x64"),
                   (330, 1500, 1200, "64x64")]
FOUR_BYTE_ROUND_SIZES = [(20, 3000, 1536, "16x32"), (100, 1500, 2560, "32x32"), (40, 5000, 768, "32x64"), (264, 3000, 2560, "64x64")]


@pytest.mark.parametrize("flags,M0,N0,K0", FOUR_BYTE_LAYOUTS)
def test_four_byte_pieces(gpu_lib, flags, M0, N0, K0):  # noqa: F811
    e = 1 if flags == abi.MMT4D_TYPE_S8S8S32 else 2
    for n, (rows, cols, row_bytes, tile) in enumerate(FOUR_BYTE_SIZES + FOUR_BYTE_ROUND_SIZES):
        pad = 16 * (n % 2) if row_bytes % 128 else 0
        run_case(gpu_lib, flags, -(-rows // M0), -(-cols // N0), row_bytes // (K0 * e), M0, N0, K0, "mmt4d_mfma_wave_k_" + tile,
                 lhs_pad=pad, rhs_pad=pad, out_pad=4 * (n % 2), accumulate=n % 3 == 1, seed=n)


def test_what_lies_behind_K_does_not_count(gpu_lib):  # noqa: F811
    import ctypes as C
    import torch
    from test_gpu_configs import mm_params
    for K0, K in ((4, 21), (1, 83), (2, 43)):
        M, N, T = 2, 3, 16
        stride = (K + 40) * T * K0
        g = torch.Generator(device="cuda").manual_seed(K)
        lhs, rhs = (torch.randn(n, stride, device="cuda", generator=g) for n in (M, N))
        a, b = (t[:, :K * T * K0].reshape(-1, K, T, K0).permute(0, 2, 1, 3).reshape(-1, K * K0).double() for t in (lhs, rhs))
        lhs[:, K * T * K0:] = float("nan")
        rhs[:, K * T * K0:] = float("inf")
        out = torch.zeros(M * N * T * T, device="cuda")
        p = mm_params(lhs.data_ptr(), rhs.data_ptr(), out.data_ptr(), M, N, K, T, T, K0, abi.MMT4D_TYPE_F32F32F32, lhs_stride=stride,
                      rhs_stride=stride, out_stride=N * T * T)
        gpu_lib.iree_uk_mmt4d_p(C.byref(p))
        assert gpu_lib.iree_uk_mi355x_last_kernel().decode() == "mmt4d_mfma_wave_k_16x16"
        got = out.view(M, N, T, T).permute(0, 2, 1, 3).reshape(M * T, N * T).double()
        assert float((got - a @ b.t()).abs().max()) < 1e-4
