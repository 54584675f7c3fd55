"""The rounding of f32 sums to a 16-bit output, and the widening of what an accumulating call finds there, value by value on the
device, bit for bit against the oracle's conversions. bf16: every sign and exponent from 1 to 254 with mantissas around every kind of
tie, overflow by rounding, subnormal sums, infinities, NaNs; all 65536 values of either output. A plain call's sum takes any f32 value
whose parts are normal (exponents from 24 on): it is hi + mid + lo, three bf16 values whose sums in any order are exact, times one.
An accumulating call's takes any: the upper half of the value is what the output holds, the lower half two products.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, mm_params  # noqa: F401

pytestmark = pytest.mark.gpu

FLAGS = abi.MMT4D_TYPE_BF16BF16BF16 | abi.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS
SLOTS, K0 = 10, 16  # values of a row: three k each
SIZES = {"wave_k": (512, 160), "block": (2048, 2080)}  # rows and columns, of 16x16x16 tiles


def tiled(x):  # [rows, cols] -> [rows / 16][cols / 16][16][16]
    r, c = x.shape
    return x.view(r // 16, 16, c // 16, 16).permute(0, 2, 1, 3).contiguous()


def product(gpu_lib, values, cols, before=None):  # noqa: F811
    """Row r, column c: values[r, c % SLOTS], rounded to bf16; added to `before` first."""
    rows, k = values.shape[0], 32
    hi = values.bfloat16()
    finite = torch.isfinite(hi.float())
    rest = torch.where(finite, values - hi.float(), torch.zeros_like(values))
    mid = rest.bfloat16()
    lhs = torch.zeros(rows, k, dtype=torch.bfloat16)
    for n, piece in enumerate((hi, mid, (rest - mid.float()).bfloat16())):
        lhs[:, n:3 * SLOTS:3] = piece
    rhs = torch.zeros(cols, k, dtype=torch.bfloat16)
    for c in range(cols):
        rhs[c, 3 * (c % SLOTS):3 * (c % SLOTS) + 3] = 1
    if not finite.all():  # (an infinity or a NaN in another slot would be multiplied by zero: one value a row)
        assert (values == values[:, :1]).logical_or(values != values).all()
        lhs[:, 3:], rhs[:], rhs[:, 0] = 0, 0, 1
    out = (torch.zeros(rows, cols, dtype=torch.bfloat16) if before is None else before).cuda()
    o, l, r = tiled(out), tiled(lhs.cuda()), tiled(rhs.cuda())
    p = mm_params(l.data_ptr(), r.data_ptr(), o.data_ptr(), rows // 16, cols // 16, k // K0, 16, 16, K0,
                  FLAGS | (0 if before is None else abi.MMT4D_ACCUMULATE))
    gpu_lib.iree_uk_mmt4d_p(C.byref(p))
    name = gpu_lib.iree_uk_mi355x_last_kernel().decode()
    got = o.cpu().view(rows // 16, cols // 16, 16, 16).permute(0, 2, 1, 3).reshape(rows, cols)
    return got.view(torch.int16).numpy().view(np.uint16), name


def narrowed(oracle_lib, x):
    f = oracle_lib.oracle_f32_to_bf16
    f.argtypes, f.restype = [C.c_float], C.c_uint16
    u, inverse = np.unique(np.ascontiguousarray(x, dtype=np.float32).view(np.uint32), return_inverse=True)
    return np.array([f(v) for v in u.view(np.float32)], dtype=np.uint16)[inverse].reshape(x.shape)


def f32(bits):
    return torch.from_numpy(np.asarray(bits, dtype=np.uint32).view(np.int32)).view(torch.float32)


@pytest.mark.parametrize("size", sorted(SIZES))
def test_finite_sums(gpu_lib, oracle_lib, size):  # noqa: F811
    rows, cols = SIZES[size]
    rng = np.random.default_rng(5)
    # Sign and exponent by row, ten mantissas: ties to even both ways, next to them, the carry into the exponent, any.
    top = (np.arange(rows, dtype=np.uint32) % 2) << 31 | ((np.arange(rows, dtype=np.uint32) // 2 * 37 % 230) + 24) << 23
    low = np.array([0, 0x8000, 0x18000, 0x7FFF, 0x8001, 0x7F8000, 0x7F7FFF, 0x7FFFFF, 0, 0], dtype=np.uint32)
    bits = top[:, None] | low[None, :]
    bits[:, 8:] |= rng.integers(0, 1 << 23, (rows, 2), dtype=np.uint32)
    values = f32(bits)
    got, name = product(gpu_lib, values, cols)
    assert name.startswith("mmt4d_mfma_wave_k" if size == "wave_k" else "mmt4d_mfma_") and ("wave_k" in name) == (size == "wave_k"), name
    want = narrowed(oracle_lib, values.numpy())
    assert np.array_equal(got, want[:, np.arange(cols) % SLOTS])


@pytest.mark.parametrize("size", sorted(SIZES))
def test_infinities_nans_and_subnormals(gpu_lib, oracle_lib, size):  # noqa: F811
    rows, cols = SIZES[size]
    special = f32([0x7F800000, 0xFF800000, 0x7FC00000, 0x7FFF0000, 0x7F7F8000, 0x00000000, 0x80000000, 0x00400000, 0x80010000, 0x007F0000])
    values = special[torch.arange(rows) % 10][:, None].expand(rows, SLOTS).contiguous()
    got, _ = product(gpu_lib, values, cols)
    want = narrowed(oracle_lib, values.numpy())[:, :1]
    # (Zeros and NaNs have the sign that the matrix pipe gives their sums.)
    signless = ((want & 0x7FFF) == 0) | ((want & 0x7FFF) > 0x7F80)
    assert np.array_equal(np.where(signless, got & 0x7FFF, got), np.broadcast_to(np.where(signless, want & 0x7FFF, want), got.shape))


@pytest.mark.parametrize("size", sorted(SIZES))
def test_every_value_of_the_output(gpu_lib, oracle_lib, size):  # noqa: F811
    rows, cols = SIZES[size]
    widen = oracle_lib.oracle_bf16_to_f32
    widen.argtypes, widen.restype = [C.c_uint16], C.c_float
    old = (np.arange(rows * cols, dtype=np.uint32) % 65536).astype(np.uint16).reshape(rows, cols)
    before = torch.from_numpy(old.view(np.int16)).view(torch.bfloat16)
    got, _ = product(gpu_lib, torch.full((rows, SLOTS), 2.0 ** -120), cols, before)
    all_values = np.arange(65536, dtype=np.uint16)
    wide = np.array([widen(int(v)) for v in all_values], dtype=np.float32)
    with np.errstate(invalid="ignore", over="ignore"):
        want = narrowed(oracle_lib, (wide + np.float32(2.0 ** -120)).astype(np.float32))[old]
    nan = (old & 0x7FFF) > 0x7F80
    assert np.array_equal(got[~nan], want[~nan])
    assert np.all(got[nan] & 0x7FFF == 0x7FFF)


def added(gpu_lib, held, rest, cols):  # noqa: F811
    """Row r, column c: held[r, s] + rest[r, s], s = c % SLOTS, rounded to bf16. `rest`: f32, at most 16 significant bits."""
    rows, k = rest.shape[0], 64
    # (Two bf16 pieces of the value times 2^64, or 2^-64, where they are normal, and back.)
    small = rest.abs() < 1
    lhs = torch.zeros(rows, k, dtype=torch.bfloat16)
    for n, scaled in ((0, torch.where(small, rest * 2.0 ** 64, torch.zeros_like(rest))),
                      (2, torch.where(small, torch.zeros_like(rest), rest * 2.0 ** -64))):
        hi = scaled.bfloat16()
        lhs[:, n:4 * SLOTS:4], lhs[:, n + 1:4 * SLOTS:4] = hi, (scaled - hi.float()).bfloat16()
    rhs = torch.zeros(cols, k, dtype=torch.bfloat16)
    for c in range(cols):
        at = 4 * (c % SLOTS)
        rhs[c, at:at + 2], rhs[c, at + 2:at + 4] = 2.0 ** -64, 2.0 ** 64
    out = held[:, torch.arange(cols) % SLOTS].cuda()
    o, l, r = tiled(out), tiled(lhs.cuda()), tiled(rhs.cuda())
    p = mm_params(l.data_ptr(), r.data_ptr(), o.data_ptr(), rows // 16, cols // 16, k // K0, 16, 16, K0, FLAGS | abi.MMT4D_ACCUMULATE)
    gpu_lib.iree_uk_mmt4d_p(C.byref(p))
    name = gpu_lib.iree_uk_mi355x_last_kernel().decode()
    got = o.cpu().view(rows // 16, cols // 16, 16, 16).permute(0, 2, 1, 3).reshape(rows, cols)
    return got.view(torch.int16).numpy().view(np.uint16), name


def bf16(bits):
    return torch.from_numpy(np.asarray(bits, dtype=np.uint16).view(np.int16)).view(torch.bfloat16)


@pytest.mark.parametrize("size", sorted(SIZES))
def test_every_exponent(gpu_lib, oracle_lib, size):  # noqa: F811
    rows, cols = SIZES[size]
    rng = np.random.default_rng(6)
    r = np.arange(rows, dtype=np.uint32)
    top = (r % 2) << 31 | (r // 2 % 254 + 1) << 23
    # (Of exponent 254 0x7F8000, a tie, and 0x7FFFFF round to infinity.)
    low = np.array([0, 0x8000, 0x18000, 0x7FFF, 0x8001, 0x7F8000, 0x7F7FFF, 0x7FFFFF, 0, 0], dtype=np.uint32)
    bits = top[:, None] | low[None, :]
    bits[:, 8:] |= rng.integers(0, 1 << 23, (rows, 2), dtype=np.uint32)
    held = bf16((bits >> 16).astype(np.uint16))
    rest = (f32(bits).double() - held.double()).float()  # (exact: the lower 16 bits)
    got, name = added(gpu_lib, held, rest, cols)
    assert ("wave_k" in name) == (size == "wave_k"), name
    want = narrowed(oracle_lib, f32(bits).numpy())
    assert (want & 0x7FFF == 0x7F80).any() and (want & 0x7F80 == 0x0080).any()
    assert np.array_equal(got, want[:, np.arange(cols) % SLOTS])


# A subnormal sum of two values that are normal is a zero of its sign.
@pytest.mark.parametrize("size", sorted(SIZES))
def test_subnormal_sums(gpu_lib, oracle_lib, size):  # noqa: F811
    rows, cols = SIZES[size]
    r = np.arange(rows * SLOTS, dtype=np.uint32).reshape(rows, SLOTS)
    held_bits = (0x0081 + r % 127 | (r // 127 % 2) << 15).astype(np.uint16)  # 2^-126 * 1.0078 .. 1.99
    held = bf16(held_bits)
    rest = torch.from_numpy(np.where(held_bits >> 15, 2.0 ** -126, -2.0 ** -126).astype(np.float32))
    sums = held.double() + rest.double()
    assert bool((sums != 0).all()) and bool((sums.abs() < 2.0 ** -126).all())
    got, _ = added(gpu_lib, held, rest, cols)
    want = narrowed(oracle_lib, sums.float().numpy())
    assert set(np.unique(want)) == {0, 0x8000}
    assert np.array_equal(got, want[:, np.arange(cols) % SLOTS])


@pytest.mark.parametrize("size", sorted(SIZES))
def test_every_value_of_an_f16_output(gpu_lib, oracle_lib, size):  # noqa: F811
    rows, cols = SIZES[size]
    widen, narrow = oracle_lib.oracle_f16_to_f32, oracle_lib.oracle_f32_to_f16
    widen.argtypes, widen.restype, narrow.argtypes, narrow.restype = [C.c_uint16], C.c_float, [C.c_float], C.c_uint16
    old = (np.arange(rows * cols, dtype=np.uint32) % 65536).astype(np.uint16).reshape(rows, cols)
    o = tiled(torch.from_numpy(old.view(np.int16)).view(torch.float16).cuda())
    l, r = (torch.zeros(n * 32, dtype=torch.float16, device="cuda") for n in (rows, cols))
    p = mm_params(l.data_ptr(), r.data_ptr(), o.data_ptr(), rows // 16, cols // 16, 2, 16, 16, K0,
                  abi.MMT4D_TYPE_F16F16F16 | abi.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS | abi.MMT4D_ACCUMULATE)
    gpu_lib.iree_uk_mmt4d_p(C.byref(p))
    got = o.cpu().view(rows // 16, cols // 16, 16, 16).permute(0, 2, 1, 3).reshape(rows, cols).view(torch.int16).numpy().view(np.uint16)
    want = np.array([narrow(np.float32(widen(int(v))) + np.float32(0)) for v in np.arange(65536)], dtype=np.uint16)[old]
    nan = (old & 0x7FFF) > 0x7C00  # (whose sign an addition may change)
    assert np.array_equal(got[~nan], want[~nan]) and np.all(got[nan] & 0x7FFF == 0x7FFF)
