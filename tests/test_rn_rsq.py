"""The correctly rounded square root, reciprocals and quotient built on v_rsq_f32 / v_rcp_f32
(csrc/cr_math.hpp): exhaustively on the CPU from every start the hardware's 1-ulp bound allows
(tests/c/rn_rsq_check.c), and on the GPU over every float of the range (tests/c/rn_gpu_check.hip)."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_refinements_are_exact(tmp_path):
    exe = str(tmp_path / "rn_rsq_check")
    subprocess.run(["gcc", "-O2", "-mfma", "-ffp-contract=off", os.path.join(HERE, "c", "rn_rsq_check.c"),
                    "-lm", "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("lo,hi", [(-96, 0), (0, 97)])
def test_every_float_on_the_gpu(gpu, lo, hi):
    import torch

    lib = ctypes.CDLL(os.path.join(HERE, "c", "librn_gpu_check.so"))
    miss = torch.zeros(3, dtype=torch.int64, device=gpu)
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.mm_rn_check(ctypes.c_uint((lo + 127) << 23), ctypes.c_uint((hi + 127) << 23),
                           ctypes.c_void_p(miss.data_ptr()), ctypes.c_void_p(stream)) == 0
    torch.cuda.synchronize()
    assert miss.tolist() == [0, 0, 0]
