"""Which f32 products are split into bf16 pieces, and in which tile, on the CPU (host_launches.py): those that the GPU tests are
made for, and none that the kernel does not cover."""
import re

import pytest

from host_launches import recorder  # noqa: F401
import test_gpu_split_f32 as gpu


def tile_of(recorder, *args, **kwargs):  # noqa: F811
    m = re.search(r"mmt4d_mfma_split_f32_(\d+x\d+)_kernelILi(\d+)E", recorder.mmt4d(gpu.F32, *args, **kwargs)[0])
    return m and (int(m[2]), m[1])


@pytest.mark.parametrize("M0,N0,K0", gpu.LAYOUTS)
@pytest.mark.parametrize("tile", ["64x64", "64x128"])
def test_gpu_problems(recorder, tile, M0, N0, K0):  # noqa: F811
    for M, N, K, options in gpu.problems(tile, M0, N0, K0):
        pads = {p: options[p] for p in ("lhs_pad", "rhs_pad", "out_pad")}
        assert tile_of(recorder, M, N, K, M0, N0, K0, **pads) == (4 if K0 == 1 else 16, tile), (M * M0, N * N0, K * K0)


def test_special_values(recorder):  # noqa: F811
    for tile, (M, N, K) in gpu.SMALL.items():
        assert tile_of(recorder, M, N, K, 16, 16, 4) == (16, tile)


# 784 x 2304 x 1920.
def test_what_it_does_not_cover(recorder):  # noqa: F811
    assert tile_of(recorder, 49, 144, 480, 16, 16, 4)
    assert not tile_of(recorder, 784, 144, 480, 1, 16, 4)             # rows that lie apart
    assert not tile_of(recorder, 196, 144, 1920, 4, 16, 1)
    assert not tile_of(recorder, 49, 144, 960, 16, 16, 2)             # 8-byte row pieces
    assert not tile_of(recorder, 49, 144, 480, 16, 16, 4, lhs_pad=2)  # 8-byte aligned rows
    assert not tile_of(recorder, 49, 144, 480, 16, 16, 4, rhs=(2 << 40) + 8)
    assert tile_of(recorder, 49, 144, 1920, 16, 16, 1, lhs_pad=4)
    assert not tile_of(recorder, 49, 144, 1920, 16, 16, 1, lhs_pad=1)


# Few chunks of K, few tiles, or many that fill the units badly: f32 multiply-adds.
@pytest.mark.parametrize("m,n,k", [(512, 512, 512), (256, 256, 256), (64, 2048, 2048), (1024, 1024, 256), (32, 4096, 4096), (2144, 496, 1968)])
def test_what_is_left_to_f32_multiply_adds(recorder, m, n, k):  # noqa: F811
    assert not tile_of(recorder, m // 16, n // 16, k // 4, 16, 16, 4)
