"""iree_uk_mi355x_last_kernel names the kernel that was launched: on the CPU (host_launches.py), the reported name against
the symbol of the launch, for every mmt4d layout over sizes that reach all kernels, and for pack and unpack."""
import random
import re

import pytest

from iree_amd import abi
from host_launches import recorder  # noqa: F401

LAYOUTS = [
    (abi.MMT4D_TYPE_S8S8S32, 8, 8, 4), (abi.MMT4D_TYPE_S8S8S32, 16, 16, 2), (abi.MMT4D_TYPE_S8S8S32, 16, 16, 64),
    (abi.MMT4D_TYPE_S8S8S32, 1, 16, 64), (abi.MMT4D_TYPE_S8S8S32, 8, 8, 1), (abi.MMT4D_TYPE_S8S8S32, 8, 8, 8),
    (abi.MMT4D_TYPE_S8S4S32, 16, 16, 32), (abi.MMT4D_TYPE_S8S4S32, 4, 16, 64), (abi.MMT4D_TYPE_F16F16F32, 16, 16, 16),
    (abi.MMT4D_TYPE_F16F16F32, 16, 16, 1), (abi.MMT4D_TYPE_BF16BF16F32, 16, 16, 8), (abi.MMT4D_TYPE_BF16BF16F32, 8, 8, 4),
    (abi.MMT4D_TYPE_BF16BF16F32, 1, 16, 2), (abi.MMT4D_TYPE_F32F32F32, 16, 16, 4), (abi.MMT4D_TYPE_F32F32F32, 16, 16, 1),
    (abi.MMT4D_TYPE_S16S16S32, 8, 16, 2), (abi.MMT4D_TYPE_F16F16F16, 16, 16, 16),
    (abi.MMT4D_TYPE_F16F16F16 | abi.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, 16, 16, 16),
    (abi.MMT4D_TYPE_BF16BF16BF16 | abi.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, 16, 16, 2)]


def name_of(symbol):
    m = re.search(r"\d(mmt4d_[a-z0-9_]+?)_kernel(I.*)?E", symbol)
    base, integers = m[1], [int(v) for v in re.findall(r"L[ib](\d+)E", m[2] or "")]
    if base == "mmt4d_wave_k":  # <type, int4 rhs, 16-bit output, piece, lhs and rhs fragments of 16 rows, ...>
        return "mmt4d_mfma_wave_k_%dx%d" % (16 * integers[4], 16 * integers[5])
    if base in ("mmt4d_mfma", "mmt4d_mfma_direct"):  # <..., lhs and rhs units of 64 rows, ...>
        return "mmt4d_mfma_%dx%d" % (64 * integers[4], 64 * integers[5])
    return {"mmt4d_mfma_split_k": "mmt4d_mfma_128x64_split_k", "mmt4d_gemv_i4": "mmt4d_gemv",
            "mmt4d_gemv_i4_resident_lhs": "mmt4d_gemv_resident_lhs"}.get(base, base)


def test_mmt4d(recorder):  # noqa: F811
    rng = random.Random(1)
    seen = set()
    for flags, M0, N0, K0 in LAYOUTS:
        for _ in range(400):
            m, n, k = (round(2 ** rng.uniform(lo, hi)) for lo, hi in ((0, 12), (4, 14), (4, 13)))
            pad = rng.choice([0, 0, 0, 16, 32])
            symbol, name = recorder.mmt4d(flags, -(-m // M0), -(-n // N0), -(-k // K0), M0, N0, K0, lhs_pad=pad, rhs_pad=pad)
            assert name == name_of(symbol), (symbol, flags, M0, N0, K0, m, n, k)
            seen.add(name)
    for M, N, K, layout, want in ((1, 896, 512, (abi.MMT4D_TYPE_BF16BF16F32, 16, 16, 8), "mmt4d_gemv_resident_lhs"),
                                  (1, 1792, 256, (abi.MMT4D_TYPE_S8S4S32, 1, 16, 32), "mmt4d_gemv_resident_lhs"),
                                  (8, 562, 512, (abi.MMT4D_TYPE_BF16BF16F32, 16, 16, 8), "mmt4d_mfma_128x64_split_k")):
        symbol, name = recorder.mmt4d(layout[0], M, N, K, *layout[1:])
        assert name == want == name_of(symbol), (symbol, name)
        seen.add(name)
    tiles = ["256x256", "256x128", "128x128", "128x64", "64x64", "64x128", "192x192", "128x192", "192x128", "256x192", "192x256",
             "128x64_split_k"] + ["wave_k_" + t for t in ("16x16", "16x32", "32x32", "32x64", "64x32", "64x64")]
    missing = {"mmt4d_" + n for n in ["gemv", "gemv_resident_lhs", "skinny", "generic"] + ["mfma_" + t for t in tiles]} - seen
    assert not missing


@pytest.mark.parametrize("flags", [0, abi.PACK_TRANSPOSE_INNER, abi.PACK_TRANSPOSE_OUTER])
@pytest.mark.parametrize("typ,t0,t1", [(abi.PACK_TYPE_I8I8, 16, 64), (abi.PACK_TYPE_BF16BF16, 16, 8), (abi.PACK_TYPE_F32F32, 16, 1),
                                       (abi.PACK_TYPE_F32F32, 6, 5)])
def test_pack(recorder, typ, t0, t1, flags):  # noqa: F811
    outer, tile = [20, 30], [t0, t1]
    if flags & abi.PACK_TRANSPOSE_OUTER:
        outer.reverse()
    if flags & abi.PACK_TRANSPOSE_INNER:
        tile.reverse()
    p = abi.PackParams()
    p.in_buffer, p.in_stride0, p.in_stride1 = 1 << 40, 30 * t1, 1
    p.out_buffer, p.out_stride0, p.out_stride1 = 2 << 40, outer[1] * t0 * t1, t0 * t1
    p.in_size0, p.in_size1 = 20 * t0, 30 * t1
    p.out_size0, p.out_size1, p.out_size2, p.out_size3 = outer + tile
    p.flags = typ | flags
    symbol, name = recorder.call("iree_uk_pack_p", p)
    kernels = {"pack_tiled": "tiled_kernel", "pack_transposing": "pack_transposing_"}
    assert kernels.get(name, "generic") in symbol, (symbol, name)
