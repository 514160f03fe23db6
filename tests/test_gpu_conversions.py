"""The hardware conversions of csrc/cr_math.hpp against what they stand for, over every float (tests/c/cvt_gpu_check.hip)."""
import ctypes
import os

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.gpu
@pytest.mark.parametrize("lo,hi", [(0x00000000, 0x7FFFFFFF), (0x80000000, 0xFFFFFFFF)])
def test_every_float(gpu, lo, hi):
    import torch

    lib = ctypes.CDLL(os.path.join(HERE, "c", "libcvt_gpu_check.so"))
    miss = torch.zeros(2, dtype=torch.int64, device=gpu)
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.mm_cvt_check(ctypes.c_uint(lo), ctypes.c_uint(hi), ctypes.c_void_p(miss.data_ptr()),
                            ctypes.c_void_p(stream)) == 0
    torch.cuda.synchronize()
    assert miss.tolist() == [0, 0]
