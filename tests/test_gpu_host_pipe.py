"""Operands in ordinary host memory pass through pinned memory in chunks (128 KiB doubling to 1 MiB, eight in turn) and
come back in pieces of 32 KiB, two halves of 4 MiB in turn; large ones are copied by several threads. The sizes lie on
both sides of each of these lines, at odd addresses and bit for bit against numpy, from one thread and from three."""
import concurrent.futures
import ctypes as C

import numpy as np
import pytest
import torch

from iree_amd import abi
from test_gpu_grid import gpu_lib  # noqa: F401

pytestmark = pytest.mark.gpu


def product(lib, M, N, K, accumulate, seed):
    print("host product", M, N, K, accumulate, flush=True)
    rng = np.random.default_rng(seed)
    lhs = rng.integers(-128, 128, M * K * 32 + 1, dtype=np.int8)[1:]
    rhs = rng.integers(-128, 128, N * K * 32 + 3, dtype=np.int8)[3:]
    guard = 64
    out = rng.integers(-1000, 1000, M * N * 256 + 2 * guard, dtype=np.int32)
    before = out.copy()
    p = abi.Mmt4dParams()
    p.lhs_buffer, p.rhs_buffer, p.out_buffer = lhs.ctypes.data, rhs.ctypes.data, out[guard:].ctypes.data
    p.lhs_stride0, p.rhs_stride0, p.out_stride0 = K * 32, K * 32, N * 256
    p.M, p.N, p.K, p.M0, p.N0, p.K0 = M, N, K, 16, 16, 2
    p.flags = abi.MMT4D_TYPE_S8S8S32 | (abi.MMT4D_ACCUMULATE if accumulate else 0)
    lib.iree_uk_mmt4d_p(C.byref(p))
    rows = lambda v, n: v.reshape(n, K, 16, 2).transpose(0, 2, 1, 3).reshape(n * 16, K * 2).astype(np.float32)  # noqa: E731
    # (|sum| <= 2048 * 2^14 = 2^25 over two halves of K, each exact in float32)
    half = K if K < 512 else K // 2
    l, r = rows(lhs, M), rows(rhs, N)
    want = sum((l[:, i:i + 2 * half] @ r[:, i:i + 2 * half].T).astype(np.int64) for i in range(0, 2 * K, 2 * half))
    want = want.reshape(M, 16, N, 16).transpose(0, 2, 1, 3).reshape(-1)
    if accumulate:
        want = want + before[guard:-guard]
    assert np.array_equal(out[guard:-guard], want), (M, N, K)
    assert np.array_equal(out[:guard], before[:guard]) and np.array_equal(out[-guard:], before[-guard:])


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 32, 3), (1, 33, 1), (8, 8, 256), (8, 9, 256), (16, 47, 512), (64, 64, 5),
                                   (65, 64, 500), (128, 64, 33), (100, 121, 1000)])
def test_lines_of_the_pipe(gpu_lib, M, N, K):  # noqa: F811
    for accumulate in (False, True, False):
        product(gpu_lib, M, N, K, accumulate, M + N + K + accumulate)


def test_several_threads(gpu_lib):  # noqa: F811
    with concurrent.futures.ThreadPoolExecutor(3) as pool:
        jobs = [pool.submit(product, gpu_lib, 64 + i, 60, 256, i % 2 == 1, i) for i in range(9)]
        for job in jobs:
            job.result()


def test_upload_behind_other_work(gpu_lib):  # noqa: F811
    # 6.7 MiB in nine chunks: the ninth reuses the first slot, whose own upload is still queued behind earlier work on the
    # caller's stream, and has to wait for it.
    a = torch.ones(8192, 8192, device="cuda")
    b = torch.empty_like(a)
    gpu_lib.iree_uk_mi355x_set_stream(torch.cuda.current_stream().cuda_stream, 0)
    for _ in range(4):
        torch.mm(a, a, out=b)
    product(gpu_lib, 100, 121, 1000, False, 5)
    torch.cuda.synchronize()
