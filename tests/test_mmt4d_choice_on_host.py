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
    ("bf16", 32, 11008, 2048, {"32x64": (9.57, 11.77), "64x64": (9.86, 12.13), "block": (10.58, 12.48)}),
    ("bf16", 64, 4096, 4096, {"32x32": (8.69, 12.70), "32x64": (10.77, 16.34), "64x32": (10.90, 16.43), "block": (17.16, 21.26)}),
    ("bf16", 96, 14336, 4096, {"block": (23.49, 31.51), "64x64": (25.34, 36.39), "32x64": (26.84, 40.35)}),
    ("bf16", 512, 4096, 4096, {"block": (22.84, 29.98), "64x64": (25.84, 36.22), "64x32": (32.44, 44.09)}),
    ("s8", 64, 14336, 4096, {"block": (12.42, 15.92), "64x64": (13.66, 14.76), "32x64": (14.27, 18.84)}),
    ("s8", 128, 4096, 14336, {"64x32": (22.03, 26.97), "32x64": (22.11, 27.09), "32x32": (27.61, 33.56), "block": (28.32, 36.02)}),
    ("s8s4", 32, 28672, 8192, {"32x64": (23.48, 25.34), "64x64": (26.08, 27.28), "16x32": (22.52, 33.90), "block": (26.98, 28.57)}),
    ("s8s4", 96, 14336, 4096, {"64x64": (14.24, 16.24), "32x64": (14.95, 18.03), "block": (16.32, 16.52)}),
    ("s8s4", 96, 11008, 2048, {"32x32": (9.08, 10.18), "block": (10.07, 10.32), "64x64": (9.95, 11.34)}),
    ("s8s4", 192, 8192, 4096, {"64x64": (14.30, 17.13), "32x64": (15.45, 18.00), "block": (16.75, 16.76)}),
    ("f16, 2-byte pieces", 64, 4096, 4096, {"32x32": (9.45, 14.99), "16x32": (12.09, 17.08), "64x32": (12.10, 17.23), "block": (33.79, 34.58)}),
    ("s8, 4-byte pieces", 128, 2048, 2048, {"32x32": (4.92, 5.50), "16x32": (5.65, 6.29), "32x64": (5.75, 6.56), "block": (6.96, 8.05)}),
    ("bf16, 8-byte pieces", 32, 14336, 4096, {"block": (19.08, 24.37), "32x64": (19.61, 24.94), "64x64": (20.61, 25.55)}),
    ("s8, 2-byte pieces", 256, 11008, 2048, {"block": (15.04, 17.74), "64x64": (19.34, 22.14), "32x32": (22.02, 27.20)}),
    ("s8, 2-byte pieces", 304, 1632, 272, {"64x32": (3.96, 4.32), "32x32": (4.11, 4.33), "block": (4.70, 5.03)}),
    ("s8, 4-byte pieces", 16, 20000, 3000, {"16x32": (11.77, 14.76), "32x32": (11.93, 15.10), "64x32": (12.92, 16.03), "block": (14.22, 16.88)}),
    ("s8, 2-byte pieces", 96, 10112, 10112, {"32x64": (27.09, 38.19), "32x32": (30.49, 42.96), "64x64": (34.90, 44.45), "block": (39.44, 40.53)}),
    ("bf16, 4-byte pieces", 16, 10112, 10112, {"32x64": (30.28, 41.46), "64x64": (30.69, 43.56), "16x16": (32.05, 44.58), "block": (39.52, 43.97)}),
    ("bf16, 4-byte pieces", 16, 20000, 3000, {"16x32": (19.15, 25.76), "32x32": (19.47, 26.00), "16x16": (19.16, 27.17), "block": (23.92, 28.90)}),
    ("s8, 2-byte pieces", 208, 5392, 1480, {"block": (10.62, 11.00), "32x32": (11.24, 12.13), "64x64": (12.13, 13.35), "32x64": (12.81, 13.90)}),
    ("s8, 2-byte pieces", 112, 8224, 2372, {"block": (13.47, 13.99), "32x32": (12.88, 14.94), "64x64": (14.61, 15.94), "64x32": (15.14, 16.88)}),
    ("bf16, 8-byte pieces", 232, 3504, 1268, {"block": (8.06, 8.88), "64x64": (9.24, 10.28), "64x32": (11.97, 13.40)}),
    ("bf16, 8-byte pieces", 72, 5648, 1776, {"block": (9.45, 10.12), "64x64": (10.27, 11.71), "32x32": (11.88, 13.63)}),
    ("s8s4", 320, 1664, 352, {"64x64": (4.28, 4.25), "32x32": (4.93, 4.85), "block": (5.11, 5.09), "32x64": (5.46, 5.40)}),
    ("f32", 64, 2048, 2048, {"16x32": (7.97, 10.13), "16x16": (8.82, 11.53), "32x32": (11.16, 12.52), "block": (36.92, 37.41)}),
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
