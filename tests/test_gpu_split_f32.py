"""f32 products whose values are split into three bf16 pieces (mmt4d_split_f32.hip), in 64x64 and in 64x128 tiles: row pieces of 4 to
64 bytes, every remainder of the number of 64-byte chunks by the wavefronts and the two steps of a loop, K ending at every place of a
chunk, ragged last tiles.

Tolerance, against a product in 64 bits: of n additions of equally large terms, each rounded by at most 2^-24 of the partial sum
(0.41 times that in the mean), the error is 0.41 * 2^-24 * sqrt(n / 2) of the result. A wavefront adds 16 values of K at a time, a
quarter of K: n = K / 64, 0.036 * sqrt(K) * 2^-24, and the last additions one each. sqrt(K) / 24 + 1 of 2^-24 leaves a
factor of 1.2 and is half of what f32 multiply-adds, rounded every two values of K, show.
"""
import ctypes as C

import pytest
import torch

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, logical, mm_params  # noqa: F401

pytestmark = pytest.mark.gpu

F32 = abi.MMT4D_TYPE_F32F32F32
LAYOUTS = [(16, 16, 4), (16, 16, 1), (8, 8, 1), (4, 16, 4), (8, 4, 8), (16, 8, 16)]  # M0, N0, K0


def problems(tile, M0, N0, K0):
    """Tiles and options of the calls: (M, N, K, options of run)."""
    sizes = {"64x64": [(432, 2044, 188), (1120, 760, 189), (688, 1324, 190), (640, 1468, 191), (300, 3196, 192), (1084, 880, 193),
                       (1344, 752, 197), (256, 4092, 199)],
             "64x128": [(784, 2304, 120), (500, 4028, 121), (1680, 1136, 122), (304, 6048, 123), (2044, 888, 125)]}[tile]
    ks = 16 // K0  # k steps of a chunk
    for n, (rows, cols, chunks) in enumerate(sizes):
        for rest in sorted({0, ks // 4, ks - 1}):
            yield (-(-rows // M0), -(-cols // N0), chunks * ks - rest,
                   dict(lhs_pad=16 * (n % 2), rhs_pad=8 * (n % 3), out_pad=4 * (n % 2), accumulate=n % 2 == 1, seed=n))


def run(gpu_lib, tile, M, N, K, M0, N0, K0, lhs_pad=0, rhs_pad=0, out_pad=0, accumulate=False, seed=0, change=None):  # noqa: F811
    """The result, the product in 64 bits and that of the magnitudes, row-major."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    l, r, o = (torch.randn(n, w, device="cuda", generator=g) for n, w in
               ((M, K * M0 * K0 + lhs_pad), (N, K * N0 * K0 + rhs_pad), (M, N * M0 * N0 + out_pad)))
    if change:
        change(l, r)
    before = o.clone()
    p = mm_params(l.data_ptr(), r.data_ptr(), o.data_ptr(), M, N, K, M0, N0, K0, F32 | (abi.MMT4D_ACCUMULATE if accumulate else 0),
                  lhs_stride=l.shape[1], rhs_stride=r.shape[1], out_stride=o.shape[1])
    gpu_lib.iree_uk_mmt4d_p(C.byref(p))
    assert gpu_lib.iree_uk_mi355x_last_kernel().decode() == "mmt4d_mfma_split_f32_" + tile

    def rows_of(x):
        return x[:, :N * M0 * N0].reshape(M, N, M0, N0).permute(0, 2, 1, 3).reshape(M * M0, N * N0).double()

    a = logical(l[:, :K * M0 * K0].contiguous(), M, K, M0, K0).double()
    b = logical(r[:, :K * N0 * K0].contiguous(), N, K, N0, K0).double()
    want = a @ b.t()
    if accumulate:
        want = want + rows_of(before)
    assert torch.equal(o[:, N * M0 * N0:], before[:, N * M0 * N0:])
    return rows_of(o), want, a.abs() @ b.abs().t() + (rows_of(before).abs() if accumulate else 0)


def bound(k):
    return 2.0 ** -24 * (1 + k ** 0.5 / 24)


@pytest.mark.parametrize("M0,N0,K0", LAYOUTS)
@pytest.mark.parametrize("tile", ["64x64", "64x128"])
def test_layouts(gpu_lib, tile, M0, N0, K0):  # noqa: F811
    for M, N, K, options in problems(tile, M0, N0, K0):
        got, want, magnitude = run(gpu_lib, tile, M, N, K, M0, N0, K0, **options)
        mean = want.square().mean().sqrt()
        error = (got - want).abs()
        assert error.square().mean().sqrt() <= bound(K * K0) * mean, (M, N, K, options)
        # Any element: the sum of K / 64 + 10 roundings of partial sums, none of which is larger than the sum of all magnitudes.
        assert (error / magnitude).max() <= (K * K0 / 64 + 10) * 2.0 ** -24, (M, N, K, options)


SMALL = {"64x64": (27, 121, 774), "64x128": (49, 144, 480)}  # in 16x16x4 tiles: 432 x 1936 x 3096, 784 x 2304 x 1920


@pytest.mark.parametrize("tile", sorted(SMALL))
def test_whole_numbers_are_exact(gpu_lib, tile):  # noqa: F811
    def whole(l, r):
        l.copy_((l * 400).round().clamp_(-1000, 1000))
        r.copy_(r.round().clamp_(-3, 3))
    got, want, _ = run(gpu_lib, tile, *SMALL[tile], 16, 16, 4, change=whole)
    assert want.abs().max() < 2 ** 24 and torch.equal(got, want)


def infinities(l, r):
    l[3, 100], r[5, 77] = float("inf"), float("-inf")


def infinity_times_zero(l, r):
    l[3, :] = 0
    l[3, 5], r[2, :] = float("inf"), 0


def nans(l, r):
    l[0, 0], r[1, 9] = float("nan"), -float("nan")


def above_the_largest_bf16(l, r):
    l[2, 33] = 3.4e38
    r.mul_(1e-3)


def sums_that_overflow(l, r):
    l[4].abs_().mul_(1e25)  # (of one sign: infinities of both would be NaN or not by the order of addition)
    r.abs_().mul_(1e18)


def large(l, r):
    l.mul_(1e18)
    r.mul_(1e17)


def small_rows(l, r):
    l[4].mul_(1e-33)
    r[6].mul_(1e-36)
    r[7].mul_(1e30)


def subnormal(l, r):
    l.mul_(1e-41)
    r.mul_(1e6)


def zeros(l, r):
    l[::2] = 0
    r[:, ::3] = -0.0


@pytest.mark.parametrize("tile", sorted(SMALL))
@pytest.mark.parametrize("change", [infinities, infinity_times_zero, nans, above_the_largest_bf16, sums_that_overflow, large, small_rows,
                                    subnormal, zeros], ids=lambda f: f.__name__)
def test_what_pieces_cannot_hold(gpu_lib, tile, change):  # noqa: F811
    got, want, _ = run(gpu_lib, tile, *SMALL[tile], 16, 16, 4, change=change)
    f32 = want.float()  # (no sum here is near the largest f32)
    assert torch.equal(torch.isnan(got), torch.isnan(f32))
    assert torch.equal(torch.isinf(got), torch.isinf(f32)) and torch.equal(got[torch.isinf(f32)], f32[torch.isinf(f32)].double())
    # Each row and column to its own scale; where f32 multiply-adds take over, to their bound: rounded every two values of K.
    finite = torch.where(torch.isfinite(f32), want, torch.zeros_like(want))
    error = torch.where(torch.isfinite(f32), got - want, torch.zeros_like(want))
    k = SMALL[tile][2] * 4
    for dim in (0, 1):
        scale = finite.square().mean(dim).sqrt() + 2.0 ** -126
        assert (error.square().mean(dim).sqrt() / scale).max() <= 4 * bound(k)
