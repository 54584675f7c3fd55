"""The block kernels' loop that takes four steps at a time (mmt4d_mfma_kernels.h, BY_FOUR): 64x64 and 128x64 tiles of 16-bit operands
with every row piece, 128x64 ones of int8 with 2-byte pieces, and the 64x128 and 128x128 tiles of an int4 rhs with one and two groups of
wavefronts. Numbers of chunks that leave it at every place of the ring (chunks modulo 8, or 4 for the 128x128 tile), just
before it is entered too, and one further on; K in whole chunks and not. That the problems take these forms is checked
in test_block_kernel_forms_on_host.py. Tolerances as in test_gpu_big_tiles: integers exact.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

S8, F16, BF16, S8S4 = abi.MMT4D_TYPE_S8S8S32, abi.MMT4D_TYPE_F16F16F32, abi.MMT4D_TYPE_BF16BF16F32, abi.MMT4D_TYPE_S8S4S32
F16_OUT16, BF16_OUT16 = abi.MMT4D_TYPE_F16F16F16, abi.MMT4D_TYPE_BF16BF16BF16

EIGHT_STAGES, FOUR_STAGES = list(range(15, 24)) + [35], list(range(11, 16)) + [35]
# Type, tile shape, block tile, groups of wavefronts, rows and columns, chunks of a group.
FORMS = [(flags, *shape, tile, 1, size, EIGHT_STAGES)
         for tile, size in (("64x64", (48, 13000)), ("128x64", (200, 8000)))
         for flags, *shape in ((F16, 16, 16, 16), (BF16, 16, 16, 8), (BF16, 8, 8, 4), (F16, 8, 16, 4), (BF16, 16, 16, 2), (F16, 4, 8, 2),
                               (BF16_OUT16, 16, 16, 16), (F16_OUT16, 8, 8, 4), (F16, 1, 16, 16))]
FORMS += [(flags, *shape, "128x64", 1, (200, 8000), EIGHT_STAGES)
          for flags, *shape in ((F16, 16, 16, 1), (BF16, 8, 8, 1), (BF16_OUT16, 16, 16, 1), (S8, 16, 16, 2), (S8, 8, 8, 2))]
FORMS += [(S8S4, *shape, tile, groups, size, chunks)
          for shape in ((16, 16, 32), (8, 4, 64))
          for tile, groups, size, chunks in (("64x128", 1, (248, 7800), EIGHT_STAGES), ("128x128", 1, (1000, 2056), FOUR_STAGES),
                                             ("64x128", 2, (304, 4104), list(range(23, 31)) + [35]), ("128x128", 2, (1000, 2056), list(range(23, 27)) + [35]))]


def problems(flags, M0, N0, K0, groups, size, chunks):
    """(M, N, K, options of run_case): for each number of chunks of a group, K whole and ending inside a chunk."""
    ks = 64 // (K0 * (1 if flags in (S8, S8S4) else 2))  # k steps of a chunk
    for count in chunks:
        for cut in sorted({0, (1 + 5 * count % (ks - 1)) if ks > 1 else 0}):
            # (two groups: an odd number of chunks where K is cut)
            K = (groups * count - (groups == 2 and cut > 0)) * ks - cut
            yield -(-size[0] // M0), -(-size[1] // N0), K, dict(accumulate=cut > 0, out_pad=4 if cut else 0, seed=count)


@pytest.mark.parametrize("form", FORMS, ids=lambda f: "t%x_%dx%dx%d_%s_%d" % f[:6])
def test_chunks(gpu_lib, form):  # noqa: F811
    flags, M0, N0, K0, tile, groups, size, chunks = form
    for M, N, K, options in problems(flags, M0, N0, K0, groups, size, chunks):
        run_case(gpu_lib, flags, M, N, K, M0, N0, K0, "mmt4d_mfma_" + tile, **options)
