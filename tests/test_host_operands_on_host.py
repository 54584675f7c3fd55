"""Calls on ordinary host memory, on the CPU with a runtime that carries out the copies (host_launches.py): what the CPU's
side of them costs, and that the bytes arrive. An accumulating product uploads its output, the kernel (which is not carried
out) leaves it alone, and it comes back."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from iree_amd import abi
from host_launches import recorder  # noqa: F401


def product(recorder, M, N, K, seed):  # noqa: F811
    """An accumulating int8 product in 16x16x2 tiles whose operands are host memory."""
    rng = np.random.default_rng(seed)
    lhs = rng.integers(-128, 128, M * K * 32, dtype=np.int8)
    rhs = rng.integers(-128, 128, N * K * 32, dtype=np.int8)
    out = rng.integers(-1000, 1000, M * N * 256, dtype=np.int32)
    before = out.copy()
    p = abi.Mmt4dParams()
    p.lhs_buffer, p.rhs_buffer, p.out_buffer = lhs.ctypes.data, rhs.ctypes.data, out.ctypes.data
    p.lhs_stride0, p.rhs_stride0, p.out_stride0 = K * 32, K * 32, N * 256
    p.M, p.N, p.K, p.M0, p.N0, p.K0 = M, N, K, 16, 16, 2
    p.flags = abi.MMT4D_TYPE_S8S8S32 | abi.MMT4D_ACCUMULATE
    recorder.lib.iree_uk_mi355x_set_stream(None, 0)
    wall, cpu = time.monotonic(), time.process_time()
    recorder.lib.iree_uk_mmt4d_p(C.byref(p))
    spent = time.monotonic() - wall, time.process_time() - cpu
    assert np.array_equal(out, before), (M, N, K)
    return spent


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 33, 1), (8, 9, 256), (16, 47, 512), (64, 64, 5), (65, 64, 500), (128, 64, 33),
                                   (100, 121, 1000), (90, 200, 900)])
def test_bytes_arrive(recorder, M, N, K):  # noqa: F811
    for seed in range(2):
        product(recorder, M, N, K, seed)


def test_from_several_threads(recorder):  # noqa: F811
    failed = []

    def calls(n):
        try:
            for i in range(3):
                product(recorder, 64 + n, 60, 256, n * 3 + i)
        except AssertionError as e:
            failed.append(e)

    threads = [threading.Thread(target=calls, args=(n,)) for n in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed


def test_a_long_product_does_not_keep_cpus_busy(recorder):  # noqa: F811
    product(recorder, 64, 64, 256, 0)  # (starts the helper threads)
    try:
        recorder.lib.recorded_set_kernel_ms(400)
        wall, cpu = product(recorder, 64, 64, 256, 1)
    finally:
        recorder.lib.recorded_set_kernel_ms(0)
    assert wall >= 0.4
    assert cpu < 0.2, (wall, cpu)


def test_pinned_memory_follows_the_calls(recorder):  # noqa: F811
    lib = recorder.lib
    lib.recorded_pinned_bytes.restype = lib.recorded_events.restype = C.c_longlong
    before = lib.recorded_pinned_bytes(), lib.recorded_events()
    seen = []

    def calls():
        for M, N, K in ((1, 1, 1), (8, 9, 256), (1, 1, 1), (64, 64, 256), (90, 200, 900), (128, 64, 33)):
            product(recorder, M, N, K, 7)
            seen.append((lib.recorded_pinned_bytes() - before[0], lib.recorded_events() - before[1]))

    t = threading.Thread(target=calls)
    t.start()
    t.join()
    kib, flags = 1 << 10, 4096
    # (0.2 MB in all; less; 5 MB; 26 MB, more than fits; less)
    assert seen == [(64 * kib + flags, 0), (256 * kib + flags, 0), (256 * kib + flags, 0), (8192 * kib + flags, 0),
                    (8192 * kib + flags, 8), (8192 * kib + flags, 8)], seen
    assert (lib.recorded_pinned_bytes(), lib.recorded_events()) == before  # given back with the thread
