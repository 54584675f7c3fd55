"""unpack into rows that end at every place inside a 16-byte vector, from tiles of up to 4 KiB, whose pieces lie alike in every
vector of a thread, and of 8 and 16 KiB, whose do not; with and without the transposes, rows a whole number of dwords apart or
not. Against the oracle byte for byte, what lies around and between the rows included."""
import ctypes as C

import numpy as np
import pytest
import torch

from iree_amd import abi, synth
from test_gpu_configs import gpu_lib  # noqa: F401

pytestmark = pytest.mark.gpu

TI, TO = abi.UNPACK_TRANSPOSE_INNER, abi.UNPACK_TRANSPOSE_OUTER


@pytest.mark.parametrize("flags", [0, TI, TO, TI | TO])
@pytest.mark.parametrize("typ,t0,t1", [
    (abi.UNPACK_TYPE_F16F16, 16, 1), (abi.UNPACK_TYPE_BF16BF16, 16, 16), (abi.UNPACK_TYPE_F16F16, 8, 2),
    (abi.UNPACK_TYPE_BF16BF16, 32, 64), (abi.UNPACK_TYPE_F16F16, 64, 64), (abi.UNPACK_TYPE_BF16BF16, 128, 64),
    (abi.UNPACK_TYPE_F32F32, 16, 4), (abi.UNPACK_TYPE_I32I32, 32, 32), (abi.UNPACK_TYPE_F32F32, 64, 32)])
def test_every_remainder(gpu_lib, oracle_lib, typ, t0, t1, flags):  # noqa: F811
    e = abi.UNPACK_ELEM_BYTES[typ]
    ve = 16 // e
    for n, cols in enumerate(list(range(1, ve + 2)) + [256 + r for r in range(ve)] + [1024 + 32 * e + r for r in range(1, ve)]):
        rows, gap, guard = (1, t0 + 1, 2 * t0 + 5)[n % 3], n % 5, 64
        o0, o1 = -(-rows // t0), -(-cols // t1)
        s0, s1 = (o1, o0) if flags & TO else (o0, o1)
        s2, s3 = (t1, t0) if flags & TI else (t0, t1)
        src = synth.uniform_int8(11, n, s0 * s1 * s2 * s3 * e)
        size = (3 + (rows - 1) * (cols + gap) + cols) * e

        def params(src_ptr, dst_ptr):
            p = abi.UnpackParams()
            p.in_buffer, p.out_buffer = src_ptr, dst_ptr + guard
            p.in_stride0, p.out_offset, p.out_stride0, p.out_stride1 = s1 * s2 * s3, 3, cols + gap, 1
            p.in_stride1 = s2 * s3
            p.in_size0, p.in_size1, p.in_size2, p.in_size3 = s0, s1, s2, s3
            p.out_size0, p.out_size1 = rows, cols
            p.flags = typ | flags
            return p

        want = np.full(size + 2 * guard, 0x77, dtype=np.int8)
        oracle_lib.oracle_unpack(C.byref(params(src.ctypes.data, want.ctypes.data)))
        d_src, d_out = torch.from_numpy(src).cuda(), torch.full((size + 2 * guard,), 0x77, dtype=torch.int8, device="cuda")
        gpu_lib.iree_uk_unpack_p(C.byref(params(d_src.data_ptr(), d_out.data_ptr())))
        assert np.array_equal(d_out.cpu().numpy(), want), (rows, cols)
