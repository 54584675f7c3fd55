"""Which mmt4d kernel the host picks, on the CPU (host_launches.py): for problems that were timed with every kernel, the one
picked is within 8 % of the best, in the geometric mean of operands that the last-level cache holds and operands from HBM."""
import math
import re

import pytest

from iree_amd import abi
from host_launches import recorder  # noqa: F401
from test_gpu_wave_k_f32_tiles import FOUR_BYTE_LAYOUTS, FOUR_BYTE_ROUND_SIZES, FOUR_BYTE_SIZES

LAYOUTS = {"bf16": (abi.MMT4D_TYPE_BF16BF16F32, 16, 16, 16), "s8": (abi.MMT4D_TYPE_S8S8S32, 16, 16, 64),
           "s8s4": (abi.MMT4D_TYPE_S8S4S32, 16, 16, 32), "s8s4, rhs tiles of 8": (abi.MMT4D_TYPE_S8S4S32, 16, 8, 32),
           "f16, 2-byte pieces": (abi.MMT4D_TYPE_F16F16F32, 16, 16, 1),
           "s8, 4-byte pieces": (abi.MMT4D_TYPE_S8S8S32, 8, 8, 4), "bf16, 8-byte pieces": (abi.MMT4D_TYPE_BF16BF16F32, 8, 8, 4),
           "bf16, 4-byte pieces": (abi.MMT4D_TYPE_BF16BF16F32, 16, 16, 2),
           "s8, 2-byte pieces": (abi.MMT4D_TYPE_S8S8S32, 16, 16, 2), "f32": (abi.MMT4D_TYPE_F32F32F32, 16, 16, 4)}

# Microseconds with operands held by the cache (150 MB in turn) and from HBM (640 MB in turn): the tiles of the kernel that
# splits K over wavefronts, and the block kernel that the problem would take.
TIMES = [
    ("bf16", 32, 11008, 2048, {"32x64": (9.16, 12.04), "block": (9.29, 12.33), "64x64": (9.36, 12.44)}),
    ("bf16", 64, 4096, 4096, {"32x32": (8.19, 12.73), "32x64": (10.28, 15.92), "64x32": (10.37, 15.95), "block": (12.23, 20.59)}),
    ("bf16", 96, 14336, 4096, {"block": (23.76, 32.71), "64x64": (25.15, 36.98), "32x64": (26.59, 40.29)}),
    ("bf16", 512, 4096, 4096, {"block": (24.62, 29.93), "64x64": (25.27, 35.74), "64x32": (31.98, 43.48)}),
    ("s8", 64, 14336, 4096, {"block": (11.68, 15.14), "64x64": (13.28, 13.76), "32x64": (13.68, 18.37)}),
    ("s8", 128, 4096, 14336, {"32x64": (21.14, 26.62), "64x32": (21.24, 26.71), "block": (24.19, 32.95), "32x32": (26.90, 32.91)}),
    ("s8s4", 32, 28672, 8192, {"32x64": (23.53, 24.44), "block": (23.80, 30.15), "16x32": (22.42, 32.52), "64x64": (27.07, 27.35)}),
    ("s8s4", 96, 14336, 4096, {"64x64": (14.45, 16.96), "block": (14.84, 16.94), "32x64": (14.32, 18.05)}),
    ("s8s4", 96, 11008, 2048, {"block": (8.80, 8.93), "32x32": (8.29, 9.63), "32x64": (9.31, 10.38), "64x64": (9.59, 10.77)}),
    ("s8s4", 192, 8192, 4096, {"block": (14.54, 15.84), "64x64": (14.81, 16.52), "32x64": (14.80, 17.18)}),
    ("f16, 2-byte pieces", 64, 4096, 4096, {"32x32": (8.81, 13.17), "32x64": (11.52, 16.57), "16x32": (11.70, 16.33), "64x32": (11.54, 16.66), "block": (29.04, 29.62)}),
    ("s8, 4-byte pieces", 128, 2048, 2048, {"32x32": (4.48, 5.00), "16x32": (5.15, 5.78), "32x64": (5.29, 6.04), "block": (5.81, 6.69)}),
    ("bf16, 8-byte pieces", 32, 14336, 4096, {"block": (18.70, 25.03), "32x64": (19.24, 24.96), "32x32": (19.52, 26.51), "64x64": (20.33, 25.92)}),
    ("s8, 2-byte pieces", 256, 11008, 2048, {"block": (14.27, 17.38), "64x64": (18.53, 21.27), "32x32": (20.95, 26.34)}),
    ("s8, 2-byte pieces", 304, 1632, 272, {"32x32": (3.92, 3.89), "64x32": (3.92, 3.90), "block": (4.62, 4.59)}),
    ("s8, 4-byte pieces", 16, 20000, 3000, {"16x32": (11.08, 14.46), "32x32": (11.43, 14.83), "16x16": (11.71, 16.29), "64x32": (12.29, 15.70), "block": (13.00, 16.62)}),
    ("s8, 2-byte pieces", 96, 10112, 10112, {"32x64": (27.31, 38.10), "block": (34.27, 37.37), "32x32": (30.29, 42.42), "64x64": (35.14, 43.99)}),
    ("bf16, 4-byte pieces", 16, 10112, 10112, {"32x64": (29.98, 40.50), "block": (29.65, 42.00), "64x64": (30.31, 42.96), "16x16": (31.66, 43.77)}),
    ("bf16, 4-byte pieces", 16, 20000, 3000, {"16x32": (19.05, 25.29), "16x16": (18.69, 26.41), "32x32": (19.44, 25.62), "block": (21.87, 28.44)}),
    ("s8, 2-byte pieces", 208, 5392, 1480, {"block": (9.56, 9.83), "32x32": (10.27, 11.53), "64x64": (11.47, 12.75), "32x64": (12.07, 13.20)}),
    ("s8, 2-byte pieces", 112, 8224, 2372, {"block": (11.66, 12.55), "32x32": (12.01, 14.03), "64x64": (13.85, 15.29), "64x32": (14.07, 15.95)}),
    ("bf16, 8-byte pieces", 232, 3504, 1268, {"block": (6.78, 8.52), "64x64": (8.66, 9.88), "64x32": (11.34, 12.86)}),
    ("bf16, 8-byte pieces", 72, 5648, 1776, {"block": (7.50, 9.75), "64x64": (9.80, 11.47), "32x32": (11.27, 12.97)}),
    ("s8s4", 320, 1664, 352, {"64x64": (4.21, 4.18), "32x32": (4.48, 4.45), "block": (4.93, 4.91), "32x64": (5.01, 4.99)}),
    # K ending inside a chunk of 64: short and long
    ("s8s4", 560, 1760, 288, {"64x64": (4.41, 4.40), "block": (5.02, 4.99)}),
    ("s8s4, rhs tiles of 8", 16, 17776, 544, {"16x32": (4.23, 4.69), "block": (4.80, 5.11)}),
    ("s8s4", 144, 6736, 1568, {"block": (7.86, 7.89), "32x64": (9.92, 10.54)}),
    ("s8s4", 352, 3120, 1568, {"block": (8.23, 8.04), "32x64": (10.61, 10.31)}),
    ("f32", 64, 2048, 2048, {"16x32": (7.45, 9.43), "16x16": (8.22, 10.93), "32x32": (10.51, 11.78), "block": (37.26, 36.91)}),
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
    ("f16, 2-byte pieces", 48), ("s8, 4-byte pieces", 32), ("bf16, 8-byte pieces", 48), ("bf16, 4-byte pieces", 32),
    ("s8, 2-byte pieces", 48), ("f32", 32), ("bf16", 48), ("s8", 999)])
def test_wave_k_looks_two_steps_ahead_with_a_long_K_only(recorder, layout, two_from):  # noqa: F811
    flags, M0, N0, K0 = LAYOUTS[layout]
    e = {"s8": 1, "f1": 2, "bf": 2, "f3": 4}[layout[:2]]
    for n in (240, 880):
        for steps in (24, 31, 32, 33, 40, 47, 48, 64, 72, 99, 100, 119, 120, 150):
            mangled, _ = recorder.mmt4d(flags, 48 // M0, n // N0, 64 * steps // (K0 * e), M0, N0, K0)
            m = re.search(r"mmt4d_wave_k_kernelILi\dELb0ELb0ELi\d+ELi(\d)ELi(\d)ELi8ELi(\d)E", mangled)
            assert m and (m[1] + m[2] != "11" or int(m[3]) == (3 if steps >= two_from else 2)), (steps, mangled)
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
