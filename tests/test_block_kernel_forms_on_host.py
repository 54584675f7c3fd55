"""Which form of the block kernels the GPU tests of one form reach, on the CPU (host_launches.py): the kernel's reported name has
the tile, its symbol the rest."""
import re

import pytest

from iree_amd import abi
from host_launches import recorder  # noqa: F401
import test_gpu_four_steps as four_steps
import test_gpu_two_groups as two_groups

NARROW = (abi.MMT4D_TYPE_F16F16F16, abi.MMT4D_TYPE_BF16BF16BF16)


def form(recorder, flags, M, N, K, M0, N0, K0, options):  # noqa: F811
    """Bytes of a row piece (16 for more), tile, stages and groups of wavefronts."""
    pads = {p: options.get(p, 0) for p in ("lhs_pad", "rhs_pad", "out_pad")}
    if flags in NARROW:
        flags |= abi.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS
    mangled, _ = recorder.mmt4d(flags, M, N, K, M0, N0, K0, **pads)
    m = re.search(r"mmt4d_mfma_direct_kernelILi\dELb\dELb\dELi(\d+)ELi(\d)ELi(\d)ELi(\d+)ELi\dELi(\d)E", mangled)
    assert m, mangled
    return int(m[1]), "%dx%d" % (64 * int(m[2]), 64 * int(m[3])), int(m[4]), int(m[5])


def test_two_groups(recorder):  # noqa: F811
    for flags, M0, N0, K0 in two_groups.SIXTEEN_BIT:
        for M, N, K, options in two_groups.sixteen_bit_problems(flags, M0, N0, K0):
            assert form(recorder, flags, M, N, K, M0, N0, K0, options) == (min(16, 2 * K0), "128x128", 4, 2), (flags, M, N, K)
    for M0, N0, K0 in two_groups.EIGHT_BIT:
        chunks = []
        for M, N, K, options in two_groups.eight_bit_problems(M0, N0, K0):
            assert form(recorder, two_groups.S8, M, N, K, M0, N0, K0, options) == (min(16, K0), "128x128", 4, 2), (M, N, K)
            chunks.append((-(-K * K0 // 64) % 2, K * K0 % 64 != 0))
        assert len(set(chunks)) == (2 if K0 == 64 else 4)  # even and odd, whole and cut
    for M0, N0, K0 in two_groups.FOUR_BIT:
        for sizes, expected in ((two_groups.WIDE, (16, "64x128", 8, 2)), (two_groups.TALL, (16, "128x128", 4, 2))):
            for M, N, K, options in two_groups.four_bit_problems(M0, N0, K0, sizes):
                assert form(recorder, two_groups.S8S4, M, N, K, M0, N0, K0, options) == expected, (M, N, K)


@pytest.mark.parametrize("case", four_steps.FORMS, ids=lambda f: "t%x_%dx%dx%d_%s_%d" % f[:6])
def test_four_steps(recorder, case):  # noqa: F811
    flags, M0, N0, K0, tile, groups, size, chunks = case
    e = 1 if flags in (four_steps.S8, four_steps.S8S4) else 2
    stages = 4 if tile == "128x128" else 8
    # The loop is entered from twice the ring's depth on, 12 chunks with four stages, and left at every place of it.
    entered = [c for c in chunks if c - 1 >= stages - 1 + 8]
    assert {c % stages for c in entered} == set(range(stages))
    for M, N, K, options in four_steps.problems(flags, M0, N0, K0, groups, size, chunks):
        assert form(recorder, flags, M, N, K, M0, N0, K0, options) == (16 if flags == four_steps.S8S4 else min(16, K0 * e), tile, stages, groups), (M, N, K)
        assert (-(-K * K0 * e // 64) + groups - 1) // groups in chunks
