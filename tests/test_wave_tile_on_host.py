"""Which products the kernel of mmt4d_wave_tile.hip takes, on the CPU (host_launches.py): those that its GPU tests are made for, and
none that it does not cover."""
import pytest

from iree_amd import abi
from host_launches import recorder  # noqa: F401
import test_gpu_wave_tile as gpu

NARROW = (abi.MMT4D_TYPE_F16F16F16, abi.MMT4D_TYPE_BF16BF16BF16)


def takes(recorder, flags, *args, **kwargs):  # noqa: F811
    if flags in NARROW:
        flags |= abi.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS
    return "mmt4d_mfma_wave_tile_kernel" in recorder.mmt4d(flags, *args, **kwargs)[0]


def pads(options):
    return {p: options.get(p, 0) for p in ("lhs_pad", "rhs_pad", "out_pad")}


@pytest.mark.parametrize("flags,M0,N0,K0", gpu.SIXTEEN_BIT)
def test_16_bit_operands(recorder, flags, M0, N0, K0):  # noqa: F811
    for M, N, K, options in gpu.sixteen_bit_problems(M0, N0, K0):
        assert takes(recorder, flags, M, N, K, M0, N0, K0, **pads(options)), (M * M0, N * N0, K * K0)


@pytest.mark.parametrize("M0,N0", gpu.FOUR_BIT)
def test_four_bit_rhs(recorder, M0, N0):  # noqa: F811
    for M, N, K, options in gpu.four_bit_problems(M0, N0):
        assert takes(recorder, gpu.S8S4, M, N, K, M0, N0, 32, **pads(options)), (M * M0, N * N0, 32 * K)


# 112 x 128 k steps of 16 bf16 in 16x16 tiles: 14 by 16 tiles of 128x128, 64 chunks.
def test_what_it_does_not_cover(recorder):  # noqa: F811
    bf16 = gpu.BF16
    assert takes(recorder, bf16, 112, 128, 128, 16, 16, 16)
    assert takes(recorder, bf16, 448, 512, 256, 4, 4, 8)
    assert not takes(recorder, bf16, 448, 128, 512, 4, 16, 4)   # 8-byte row pieces
    assert not takes(recorder, bf16, 112, 128, 64, 16, 16, 32)  # 64-byte ones: four lanes touch two lines
    assert not takes(recorder, bf16, 1792, 128, 128, 1, 16, 16)  # rows that lie apart
    assert not takes(recorder, bf16, 112, 128, 128, 16, 16, 16, lhs_pad=4)  # 8-byte aligned rows
    assert not takes(recorder, bf16, 112, 128, 128, 16, 16, 16, rhs=(2 << 40) + 8)
    assert takes(recorder, gpu.S8S4, 31, 137, 91, 16, 16, 32)
    assert not takes(recorder, gpu.S8S4, 31, 137, 46, 16, 16, 64)
    assert not takes(recorder, abi.MMT4D_TYPE_S8S8S32, 112, 128, 128, 16, 16, 32)
    assert not takes(recorder, abi.MMT4D_TYPE_F32F32F32, 112, 128, 256, 16, 16, 4)


# Where the lines lie: tiles, chunks of K, bytes of the operands.
def test_where_it_is_taken(recorder):  # noqa: F811
    def bf16(tile_rows, tile_cols, chunks):
        return takes(recorder, gpu.BF16, 8 * tile_rows, 8 * tile_cols, 2 * chunks, 16, 16, 16)
    assert [bf16(r, c, 64) for r, c in ((11, 18), (10, 20), (8, 31), (10, 25), (16, 16))] == [False, True, True, False, False]
    assert [bf16(12, 18, chunks) for chunks in (63, 64, 204, 205)] == [False, True, True, False]  # 48 MiB

    def i4(rows, cols, k):
        return takes(recorder, gpu.S8S4, -(-rows // 16), -(-cols // 16), k // 32, 16, 16, 32)
    # 64x64 tiles that fit a round, 64x128 ones that do.
    assert [i4(304, n, 3360) for n in (3264, 3280)] == [False, True]
    assert [i4(320, 3424, 3360), i4(224, 4944, 2592), i4(160, 6160, 4128), i4(144, 5712, 4640)] == [True, True, False, False]


# int4: not where the units hold all tiles of 32x64 at once, two workgroups each.
def test_four_bit_rhs_of_one_round_of_small_tiles(recorder):  # noqa: F811
    def i4(rows, cols, k):
        return takes(recorder, gpu.S8S4, rows // 16, cols // 16, k // 32, 16, 16, 32)
    assert not any(i4(*size) for size in [(480, 2144, 7872), (608, 1632, 2528), (784, 1264, 5888), (2704, 384, 2656), (224, 4640, 7232)])
    assert [i4(480, n, 4096) for n in (2176, 2192)] == [False, True]  # 15 rows of 34 and 35 tiles
