"""Which kernel a bf16 Hessian call takes, read from the workspace it asks for (the few-rows
kernel asks for none, the row splits for their partial tiles). No GPU is needed."""
import pytest

from perm_amd import _lib


# measured, us a call, few-rows kernel / row splits
FEW = [(2048, 1024, 1),    # 17 / 31
       (12288, 1024, 1),   # 51 / 54
       (49152, 256, 1),    # 138 / 218
       (64, 1400, 1),      # 13 / 60
       (14000, 896, 1),    # 52 / 58
       (4096, 512, 6),     # 37 / 42
       (8192, 512, 4),     # 47 / 51
       (2048, 256, 25),    # 55 / 60
       (32768, 64, 64)]    # 122 / 165
SPLIT = [(8192, 512, 6),     # 64 / 48: six jobs' rows, not one's
         (24576, 512, 3),    # 102 / 67
         (8192, 256, 25),    # 74 / 61
         (49152, 256, 5),    # 145 / 95
         (16384, 256, 12),   # 73 / 61
         (16384, 1024, 1),   # 66 / 61
         (14000, 880, 1),    # 70 / 58: rows of 1760 bytes end inside a 128-byte line
         (196608, 64, 1),    # 482 / 316: one workgroup walks every row
         (65536, 32, 1),     # 162 / 138
         (65536, 8, 1),      # 160 / 71
         (393216, 32, 1),    # 953 / 185
         (1572864, 8, 1)]    # 3787 / 175


@pytest.mark.parametrize("N,d,jobs,few", [(*c, True) for c in FEW] + [(*c, False) for c in SPLIT])
def test_bf16_call_takes_the_faster_kernel(N, d, jobs, few):
    ws = _lib.load(require_gpu=False).cp_hess_ws_bytes(jobs, 1, N, d)
    assert (ws == 0) == few, ws
