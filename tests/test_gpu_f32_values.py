"""What an f32 product is, whichever kernel runs it: a product of two values is rounded to f32 once, as a multiply-add does it, and
a row's bits depend on that row and the rhs alone, not on what other rows of its tile hold (padding that a caller never wrote
among them). Infinities, NaNs, subnormals, values and products near the ends of the range.

Tolerance, against a product in 64 bits: f32 MFMAs add two values of K at a time, K / 2 additions in a row at most, each rounded by
0.41 * 2^-24 of the partial sum in the mean. Terms of either sign at random make a result of the size of the root of the sum of their
squares, and partial sums of half of its square in the mean: 0.41 * 2^-24 * sqrt(K / 4) of that size. Wavefronts that share K have
shorter rows of additions: a third to two thirds of it is seen.
"""
import ctypes as C

import pytest
import torch

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, mm_params  # noqa: F401

pytestmark = pytest.mark.gpu

# Rows, columns, K, K0: tiles of 48x80 and 80x48 over eight wavefronts, 4-byte row pieces, block kernels, few rows.
SIZES = [(432, 1936, 3096, 4), (784, 2304, 1920, 4), (432, 1936, 3096, 1), (1024, 2048, 2048, 4), (528, 6480, 612, 4), (48, 80, 512, 4),
         (1040, 4112, 72, 1)]


def run(gpu_lib, a, b, K0):  # noqa: F811
    """a @ b.T by the library, in tiles of 16 x 16 x K0."""
    def tiled(x):
        return x.view(x.shape[0] // 16, 16, x.shape[1] // K0, K0).permute(0, 2, 1, 3).contiguous()
    l, r = tiled(a), tiled(b)
    o = torch.zeros(a.shape[0] // 16, b.shape[0] // 16, 16, 16, device="cuda")
    p = mm_params(l.data_ptr(), r.data_ptr(), o.data_ptr(), a.shape[0] // 16, b.shape[0] // 16, a.shape[1] // K0, 16, 16, K0,
                  abi.MMT4D_TYPE_F32F32F32)
    gpu_lib.iree_uk_mmt4d_p(C.byref(p))
    return o.permute(0, 2, 1, 3).reshape(a.shape[0], b.shape[0])


def operands(rows, cols, k):
    g = torch.Generator(device="cuda").manual_seed(rows + cols + k)
    return [torch.randn(n, k, device="cuda", generator=g) for n in (rows, cols)]


@pytest.mark.parametrize("rows,cols,k,K0", SIZES)
def test_one_product_a_sum_is_rounded_once(gpu_lib, rows, cols, k, K0):  # noqa: F811
    a, b = operands(rows, cols, k)
    at = torch.arange(rows, device="cuda") * 37 % k
    only = torch.zeros_like(a)
    only[torch.arange(rows, device="cuda"), at] = a[torch.arange(rows, device="cuda"), at]
    want = a[torch.arange(rows, device="cuda"), at][:, None] * b[:, at].t()
    assert torch.equal(run(gpu_lib, only, b, K0), want)


@pytest.mark.parametrize("rows,cols,k,K0", SIZES)
@pytest.mark.parametrize("value", [1e-35, 1e-41, float("inf"), float("nan"), 3.4e38])
def test_other_rows_keep_their_bits(gpu_lib, rows, cols, k, K0, value):  # noqa: F811
    a, b = operands(rows, cols, k)
    before = run(gpu_lib, a, b, K0)
    a[5, 3] = a[rows - 1, k - 1] = value
    b[7, 2] = value
    after = run(gpu_lib, a, b, K0)
    before, after = (x.view(torch.int32).clone() for x in (before, after))
    for x in (before, after):
        x[5] = x[rows - 1] = x[:, 7] = 0
    assert torch.equal(before, after)


def infinities(a, b):
    a[3, 100], b[5, 47] = float("inf"), float("-inf")


def infinity_times_zero(a, b):
    a[3, :] = 0
    a[3, 5], b[2, :] = float("inf"), 0


def nans(a, b):
    a[0, 0], b[1, 9] = float("nan"), -float("nan")


def the_largest(a, b):
    a[2, 33] = 3.4e38
    b.mul_(1e-3)


def a_sum_that_overflows(a, b):
    a[4].abs_().mul_(1e25)  # (of one sign: infinities of both would be NaN or not by the order of addition)
    b[9].abs_().mul_(1e18)


def large(a, b):
    a.mul_(1e18)
    b.mul_(1e17)


def small_products(a, b):  # about 2^-120, of values that are not small themselves
    a.mul_(1e-18)
    b.mul_(1e-18)


def small_rows(a, b):
    a[4].mul_(1e-33)
    b[6].mul_(1e-36)
    b[7].mul_(1e30)


def subnormal(a, b):
    a.mul_(1e-41)
    b.mul_(1e6)


def zeros(a, b):
    a[::2] = 0
    b[:, ::3] = -0.0


@pytest.mark.parametrize("rows,cols,k,K0", SIZES[:4])
@pytest.mark.parametrize("change", [infinities, infinity_times_zero, nans, the_largest, a_sum_that_overflows, large, small_products, small_rows,
                                    subnormal, zeros], ids=lambda f: f.__name__)
def test_ends_of_the_range(gpu_lib, rows, cols, k, K0, change):  # noqa: F811
    a, b = operands(rows, cols, k)
    change(a, b)
    got, want = run(gpu_lib, a, b, K0).double(), a.double() @ b.double().t()
    f32 = want.float()  # (no sum here is near the largest f32)
    assert torch.equal(torch.isnan(got), torch.isnan(f32))
    assert torch.equal(torch.isinf(got), torch.isinf(f32)) and torch.equal(got[torch.isinf(f32)], f32[torch.isinf(f32)].double())
    bound = 0.41 * 2.0 ** -24 * (k / 4) ** 0.5
    size = (a.double().square() @ b.double().square().t()).sqrt() + 2.0 ** -149 * k ** 0.5 / bound  # (below, f32 has no more bits)
    error = torch.where(torch.isfinite(f32), (got - want) / size, torch.zeros_like(want))
    for dim in (0, 1):  # each row and column to its own size
        assert error.square().mean(dim).sqrt().max() <= bound
