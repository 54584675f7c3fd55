"""Which mmt4d kernel the host picks, on the CPU (host_launches.py): for problems that were timed with every kernel, the one
picked is within 8 % of the best, in the geometric mean of operands that the last-level cache holds and operands from HBM."""
import math
import re

import pytest

from iree_amd import abi
from host_launches import recorder  # noqa: F401
from test_gpu_wave_k_f32_tiles import FOUR_BYTE_LAYOUTS, FOUR_BYTE_ROUND_SIZES, FOUR_BYTE_SIZES

LAYOUTS = {"bf16": (abi.MMT4D_TYPE_BF16BF16F32, 16, 16, 16), "s8": (abi.MMT4D_TYPE_S8S8S32, 16, 16, 64),
           "s8s4": (abi.MMT4D_TYPE_S8S4S32, 16, 16, 32), "f16, 2-byte pieces": (abi.MMT4D_TYPE_F16F16F32, 16, 16, 1),
           "s8, 4-byte pieces": (abi.MMT4D_TYPE_S8S8S32, 8, 8, 4), "bf16, 8-byte pieces": (abi.MMT4D_TYPE_BF16BF16F32, 8, 8, 4),
           "bf16, 4-byte pieces": (abi.MMT4D_TYPE_BF16BF16F32, 16, 16, 2),
           "s8, 2-byte pieces": (abi.MMT4D_TYPE_S8S8S32, 16, 16, 2), "f32": (abi.MMT4D_TYPE_F32F32F32, 16, 16, 4)}

# Microseconds with operands held by the cache (150 MB in turn) and from HBM (640 MB in turn): the tiles of the kernel that
# splits K over wavefronts, and the block kernel that the problem would take.
TIMES = [
    ("bf16", 32, 11008, 2048, {"32x64": (9.8, 12.5), "64x64": (10.0, 12.8), "16x32": (10.4, 13.8), "block": (11.9, 13.2)}),
    ("bf16", 64, 4096, 4096, {"32x32": (9.2, 13.1), "16x32": (11.2, 16.0), "32x64": (11.0, 16.5), "block": (19.7, 21.0)}),
    ("bf16", 96, 14336, 4096, {"block": (23.9, 32.6), "64x64": (26.6, 38.4), "32x64": (27.5, 40.7)}),
    ("bf16", 512, 4096, 4096, {"block": (24.5, 30.0), "64x64": (26.4, 35.1), "64x32": (32.1, 42.4)}),
    ("s8", 64, 14336, 4096, {"64x64": (14.2, 14.7), "block": (12.8, 16.5), "32x64": (14.7, 19.3)}),
    ("s8", 128, 4096, 14336, {"32x64": (22.2, 26.9), "64x32": (22.1, 27.3), "32x32": (27.8, 33.1), "block": (32.0, 35.9)}),
    ("s8s4", 32, 28672, 8192, {"32x64": (25.4, 26.1), "16x32": (24.1, 33.9), "64x64": (28.4, 28.8), "block": (27.2, 30.7)}),
    ("s8s4", 96, 14336, 4096, {"block": (16.2, 16.3), "64x64": (15.8, 17.9), "32x64": (16.2, 19.3)}),
    ("s8s4", 96, 11008, 2048, {"block": (10.2, 10.3), "32x64": (10.8, 11.8), "64x64": (10.4, 12.4)}),
    ("s8s4", 192, 8192, 4096, {"64x64": (15.3, 17.9), "block": (16.6, 16.7), "32x64": (16.6, 18.7)}),
    ("f16, 2-byte pieces", 64, 4096, 4096, {"32x32": (10.8, 13.9), "16x32": (13.3, 16.7), "64x32": (14.0, 17.5), "block": (37.6, 37.9)}),
    ("s8, 4-byte pieces", 128, 2048, 2048, {"32x32": (5.6, 5.9), "16x32": (6.1, 6.4), "32x64": (6.5, 6.9), "block": (7.8, 7.9)}),
    ("bf16, 8-byte pieces", 32, 14336, 4096, {"32x64": (20.5, 25.2), "block": (19.9, 26.0), "64x64": (21.8, 26.6)}),
    ("s8, 2-byte pieces", 256, 11008, 2048, {"block": (15.5, 17.6), "64x64": (21.2, 23.8), "64x32": (28.1, 31.4)}),
    ("s8, 2-byte pieces", 304, 1632, 272, {"64x32": (4.0, 4.1), "64x64": (4.7, 4.9), "block": (4.8, 5.0)}),
    ("s8, 4-byte pieces", 16, 20000, 3000, {"16x32": (12.4, 15.2), "16x16": (13.3, 17.0), "block": (14.5, 17.4)}),
    ("s8, 2-byte pieces", 96, 10112, 10112, {"32x64": (31.5, 39.0), "block": (44.3, 44.6), "64x64": (42.0, 48.4)}),
    ("bf16, 4-byte pieces", 16, 10112, 10112, {"32x64": (41.7, 41.7), "16x32": (47.6, 47.6), "16x16": (45.1, 45.0), "block": (48.3, 48.1)}),
    ("bf16, 4-byte pieces", 16, 20000, 3000, {"16x32": (20.8, 25.9), "16x16": (20.6, 28.0), "block": (24.4, 29.5)}),
    ("f32", 64, 2048, 2048, {"16x32": (10.2, 10.8), "16x16": (12.2, 13.0), "32x32": (15.9, 16.7), "block": (37.4, 37.5)}),
]


def kernel_of(mangled):
    """"block", or the tile of the kernel that splits K over wavefronts."""
    m = re.search(r"mmt4d_wave_k_kernelILi\dELb\dELb\dELi\d+ELi(\d)ELi(\d)E", mangled)
    if m:
        return "%dx%d" % (16 * int(m[1]), 16 * int(m[2]))
    assert "mmt4d_mfma" in mangled, mangled
    return "block"


@pytest.mark.parametrize("layout,m,n,k,times", TIMES, ids=lambda v: "times" if isinstance(v, dict) else str(v))
def test_the_kernel_picked_is_among_the_best(recorder, layout, m, n, k, times):  # noqa: F811
    flags, M0, N0, K0 = LAYOUTS[layout]
    mangled, _ = recorder.mmt4d(flags, m // M0, n // N0, k // K0, M0, N0, K0)
    picked = kernel_of(mangled)
    assert picked in times, mangled
    mean = {name: math.sqrt(held * hbm) for name, (held, hbm) in times.items()}
    assert mean[picked] <= 1.08 * min(mean.values()), (picked, mean)


def streams(mangled):
    """Whether a matrix-vector kernel, or the one that splits K over wavefronts, reads the rhs past the caches."""
    m = (re.search(r"mmt4d_gemv_kernelILi\dELi\d+ELi\d+ELi\d+ELb(\d)E", mangled) or
         re.search(r"mmt4d_gemv_i4_kernelILi\d+ELi\d+ELi\d+ELb(\d)E", mangled) or
         re.search(r"mmt4d_skinny_kernelILi\dELi\dELi\dELi\dELi\d+ELb(\d)ELb\dE", mangled) or
         re.search(r"mmt4d_wave_k_kernelILi\dELb\dELb\dELi16ELi\dELi\dELi\dELi\dELb(\d)E", mangled))
    assert m, mangled
    return m[1] == "1"


# Weights are taken to come from HBM above 48 MiB, whichever kernel reads them.
@pytest.mark.parametrize("flags,M,M0,N0,K0,n,k,bits", [
    (abi.MMT4D_TYPE_BF16BF16F32, 1, 1, 16, 8, 6144, 4096, 16), (abi.MMT4D_TYPE_S8S8S32, 1, 1, 16, 64, 12288, 4096, 8),
    (abi.MMT4D_TYPE_S8S4S32, 1, 4, 16, 32, 12288, 8192, 4), (abi.MMT4D_TYPE_S8S8S32, 1, 1, 16, 2, 12288, 4096, 8),
    (abi.MMT4D_TYPE_BF16BF16F32, 1, 4, 16, 2, 6144, 4096, 16), (abi.MMT4D_TYPE_F32F32F32, 1, 2, 16, 1, 6144, 2048, 32),
    (abi.MMT4D_TYPE_BF16BF16F32, 2, 16, 16, 16, 6144, 4096, 16), (abi.MMT4D_TYPE_S8S4S32, 2, 16, 16, 32, 24576, 4096, 4)])
def test_one_rule_for_weights_from_hbm(recorder, flags, M, M0, N0, K0, n, k, bits):  # noqa: F811
    assert n * k * bits // 8 <= 48 << 20
    assert not streams(recorder.mmt4d(flags, M, n // N0, k // K0, M0, N0, K0)[0])
    n += n // 16
    assert n * k * bits // 8 > 48 << 20
    assert streams(recorder.mmt4d(flags, M, n // N0, k // K0, M0, N0, K0)[0])


def test_narrow_tiles_bound_by_the_vector_alu_stream_only_what_no_cache_holds(recorder):  # noqa: F811
    s8 = abi.MMT4D_TYPE_S8S8S32
    assert not streams(recorder.mmt4d(s8, 1, 14336 // 16, 4096 // 2, 4, 16, 2)[0])
    assert streams(recorder.mmt4d(s8, 1, 28672 // 16, 8192 // 2, 4, 16, 2)[0])
    # No more tile rows than compute units: eight wavefronts a tile row, through the caches.
    assert "ELi8ELi8ELb0E" in recorder.mmt4d(s8, 1, 4096 // 16, 14336 // 2, 2, 16, 2)[0]


def test_block_kernels_have_the_deep_ring_for_operands_from_hbm(recorder):  # noqa: F811
    bf16 = abi.MMT4D_TYPE_BF16BF16F32
    for n, stages in ((11264, 4), (13312, 10)):  # 46 and 54 MiB with 192 rows
        assert "ELi2ELi2ELi%dE" % stages in recorder.mmt4d(bf16, 12, n // 16, 2048 // 16, 16, 16, 16)[0]


# Steps in flight, one more than those ahead, for one fragment either way (mmt4d_wave_k_kernels.h): with 45 tiles and with 165.
@pytest.mark.parametrize("layout,two_from", [
    ("f16, 2-byte pieces", (120, 100)), ("s8, 4-byte pieces", (120, 100)), ("bf16, 8-byte pieces", (120, 100)),
    ("bf16, 4-byte pieces", (120, 100)), ("s8, 2-byte pieces", (120, 100)), ("f32", (120, 100)), ("bf16", (48, 48)), ("s8", (999, 999))])
def test_wave_k_looks_two_steps_ahead_with_a_long_K_only(recorder, layout, two_from):  # noqa: F811
    flags, M0, N0, K0 = LAYOUTS[layout]
    e = {"s8": 1, "f1": 2, "bf": 2, "f3": 4}[layout[:2]]
    for n, threshold in zip((240, 880), two_from):
        for steps in (24, 33, 40, 47, 48, 64, 72, 99, 100, 119, 120, 150):
            mangled, _ = recorder.mmt4d(flags, 48 // M0, n // N0, 64 * steps // (K0 * e), M0, N0, K0)
            m = re.search(r"mmt4d_wave_k_kernelILi\dELb0ELb0ELi\d+ELi(\d)ELi(\d)ELi8ELi(\d)E", mangled)
            assert m and (m[1] + m[2] != "11" or int(m[3]) == (3 if steps >= threshold else 2)), (steps, mangled)
            assert n > 240 or m[1] + m[2] == "11", (steps, mangled)


# 4-byte row pieces are loaded one at a time, but through LDS where 16 rows are four tiles a multiple of 512 bytes apart: of the
# rhs always, of the lhs unless there are more fragments of an rhs in 16-row tiles. (The last template argument; the tile is
# the one that test_gpu_wave_k_f32_tiles.py expects.)
@pytest.mark.parametrize("flags,M0,N0,K0", FOUR_BYTE_LAYOUTS)
def test_four_byte_pieces_pass_through_lds_where_rows_share_memory_channels(recorder, flags, M0, N0, K0):  # noqa: F811
    e = 1 if flags == abi.MMT4D_TYPE_S8S8S32 else 2
    if flags == abi.MMT4D_TYPE_F16F16F16:
        flags |= abi.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS
    for rows, cols, row_bytes, tile in FOUR_BYTE_SIZES + FOUR_BYTE_ROUND_SIZES:
        mangled, kernel = recorder.mmt4d(flags, -(-rows // M0), -(-cols // N0), row_bytes // (K0 * e), M0, N0, K0)
        assert kernel == "mmt4d_mfma_wave_k_" + tile
        pieces = re.search(r"ELi4ELi\dELi\dELi8ELi\dELb0ELb(\d)E", mangled)[1] == "1"
        round_rows = row_bytes % 128 == 0 and (N0 == 4 or (M0 == 4 and not (N0 == 16 and tile in ("16x32", "32x64"))))
        assert pieces == (not round_rows), (rows, cols, row_bytes, mangled)


def skinny_form(mangled):
    """Lhs rows, wavefronts, blocks of 1 KiB in flight in each and whether the rhs is streamed, of the few-row kernel."""
    m = re.search(r"mmt4d_skinny_kernelILi\dELi\dELi(\d)ELi(\d)ELi(\d+)ELb(\d)E", mangled)
    assert m, mangled
    return int(m[1]), int(m[2]), int(m[3]), m[4] == "1"


# Two int8 rows, at most a tile row a unit and long ones: 8 KiB in flight for a packed lhs, 4 KiB otherwise.
def test_two_int8_rows(recorder):  # noqa: F811
    s8 = abi.MMT4D_TYPE_S8S8S32
    assert skinny_form(recorder.mmt4d(s8, 1, 200, 4200, 2, 16, 2)[0]) == (2, 8, 8, False)
    assert skinny_form(recorder.mmt4d(s8, 2, 200, 4200, 1, 16, 2)[0]) == (2, 8, 4, False)
    assert skinny_form(recorder.mmt4d(s8, 1, 200, 4200, 2, 16, 2, lhs=(1 << 40) + 2)[0]) == (2, 8, 4, False)


# One row from HBM, more than two tile rows a unit: eight wavefronts for tiles of 64 to 96 and 128 to 144 KiB, however far apart
# the tile rows lie.
@pytest.mark.parametrize("flags,K0,e", [(abi.MMT4D_TYPE_BF16BF16F32, 2, 2), (abi.MMT4D_TYPE_S8S8S32, 2, 1), (abi.MMT4D_TYPE_F32F32F32, 1, 4),
                                        (abi.MMT4D_TYPE_F16F16F32, 1, 2)])
def test_one_row_from_hbm(recorder, flags, K0, e):  # noqa: F811
    for tile_kib, eight in ((50, False), (63, False), (64, True), (65, True), (95, True), (96, False), (127, False), (128, True), (130, True),
                            (143, True), (144, False), (192, False), (256, False)):
        K = tile_kib * 1024 // (16 * K0 * e)
        for steps_off in (0, 1, 3):
            for pad in (0, 16, 1024):
                form = skinny_form(recorder.mmt4d(flags, 1, 1100, K + steps_off, 1, 16, K0, rhs_pad=pad)[0])
                assert form == ((1, 8, 4, True) if eight else (1, 4, 12, True)), (tile_kib, steps_off, pad, form)


# Five rows and more have a ring of two blocks, int16 from HBM one of four; int4 in 1-byte pieces has four wavefronts always.
def test_five_to_eight_rows(recorder):  # noqa: F811
    s16, u4, i4 = abi.MMT4D_TYPE_S16S16S32, abi.MMT4D_TYPE_S16U4S32, abi.MMT4D_TYPE_S8S4S32
    assert skinny_form(recorder.mmt4d(s16, 1, 900, 2048, 8, 16, 2)[0]) == (8, 4, 4, True)
    assert skinny_form(recorder.mmt4d(s16, 1, 900, 800, 8, 16, 2)[0]) == (8, 4, 2, False)
    assert skinny_form(recorder.mmt4d(s16, 1, 200, 2048, 8, 16, 2)[0]) == (8, 8, 2, False)
    assert skinny_form(recorder.mmt4d(s16, 1, 900, 4096, 8, 8, 2)[0]) == (8, 4, 4, True)
    assert skinny_form(recorder.mmt4d(u4, 1, 200, 512, 8, 32, 8)[0]) == (8, 8, 2, False)
    for M, M0 in ((1, 8), (5, 1), (2, 8), (2, 4)):
        assert skinny_form(recorder.mmt4d(i4, M, 64, 512, M0, 16, 2)[0]) == (8, 4, 2, False)
    assert skinny_form(recorder.mmt4d(i4, 1, 64, 512, 4, 16, 2)[0]) == (4, 8, 4, False)
    # the rest of nine rows is a slab of its own
    assert skinny_form(recorder.mmt4d(i4, 9, 64, 512, 1, 16, 2)[0])[:2] == (1, 8)
