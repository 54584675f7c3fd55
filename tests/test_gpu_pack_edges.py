"""pack of rows that end at every place inside a 16-byte vector, and of rows shorter than one: element sizes 1, 2 and 4,
with and without the transposes (the plain and both transposing kernels), at every alignment of the rows, with a padding
value whose bytes differ. Against the oracle byte for byte, what lies around the destination included."""
import ctypes as C

import numpy as np
import pytest
import torch

from iree_amd import abi, synth
from test_gpu_configs import gpu_lib  # noqa: F401

pytestmark = pytest.mark.gpu

TI, TO = abi.PACK_TRANSPOSE_INNER, abi.PACK_TRANSPOSE_OUTER


@pytest.mark.parametrize("typ,t0,t1,flags", [
    (abi.PACK_TYPE_I8I8, 16, 64, 0), (abi.PACK_TYPE_I8I8, 8, 4, TO), (abi.PACK_TYPE_I8I8, 64, 16, TI | TO),
    (abi.PACK_TYPE_I8I8, 2, 16, TI), (abi.PACK_TYPE_I8I8, 4, 8, TI | TO), (abi.PACK_TYPE_BF16BF16, 16, 8, 0),
    (abi.PACK_TYPE_F16F16, 16, 1, TO), (abi.PACK_TYPE_BF16BF16, 16, 16, TI | TO), (abi.PACK_TYPE_F16F16, 8, 16, TI),
    (abi.PACK_TYPE_F32F32, 16, 4, 0), (abi.PACK_TYPE_I32I32, 8, 8, TI | TO)])
def test_every_remainder(gpu_lib, oracle_lib, typ, t0, t1, flags):  # noqa: F811
    e = abi.PACK_ELEM_BYTES[typ]
    ve = 16 // e
    for n, cols in enumerate(list(range(1, 2 * ve + 2)) + [256 + r for r in range(ve)] + [1024 // e + 1]):
        rows, gap, guard = (1, t0 + 1, 37)[n % 3], n % 5, 64
        o0, o1 = -(-rows // t0), -(-cols // t1)
        s0, s1 = (o1, o0) if flags & TO else (o0, o1)
        s2, s3 = (t1, t0) if flags & TI else (t0, t1)
        # The input ends with its last row's last element: nothing behind it belongs to the call.
        src = synth.uniform_int8(7, n, (3 + (rows - 1) * (cols + gap) + cols) * e)
        size = s0 * s1 * s2 * s3 * e

        def params(src_ptr, dst_ptr):
            p = abi.PackParams()
            p.in_buffer, p.out_buffer = src_ptr, dst_ptr + guard
            p.in_offset, p.in_stride0, p.in_stride1 = 3, cols + gap, 1
            p.out_stride0, p.out_stride1 = s1 * s2 * s3, s2 * s3
            p.in_size0, p.in_size1 = rows, cols
            p.out_size0, p.out_size1, p.out_size2, p.out_size3 = s0, s1, s2, s3
            p.padding_value = 0xDEADBEA5
            p.flags = typ | flags
            return p

        want = np.full(size + 2 * guard, 0x77, dtype=np.int8)
        oracle_lib.oracle_pack(C.byref(params(src.ctypes.data, want.ctypes.data)))
        d_src, d_out = torch.from_numpy(src).cuda(), torch.full((size + 2 * guard,), 0x77, dtype=torch.int8, device="cuda")
        gpu_lib.iree_uk_pack_p(C.byref(params(d_src.data_ptr(), d_out.data_ptr())))
        assert np.array_equal(d_out.cpu().numpy(), want), (rows, cols)
