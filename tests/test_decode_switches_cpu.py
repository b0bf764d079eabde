"""Environment switches of the decode steps' attention that multiplies with its output projection (vy_dec_attn_out of
vyomai_amd/csrc/vy_decode.hip): which calls it leaves to other kernels, and what becomes of a launch that fails.  A
machine without a GPU shows it, where no launch succeeds."""
import os
import subprocess
import sys

import pytest
import torch

CHILD = """
import ctypes as C, sys
p, i, l, f = C.c_void_p, C.c_int, C.c_int64, C.c_float
lib = C.CDLL(sys.argv[1])
go = lib._Z15vy_dec_attn_outPKvS0_S0_lllS0_PfliiillPKifP12ihipStream_t
go.argtypes, go.restype = [p, p, p, l, l, l, p, p, l, i, i, i, l, l, p, f, p], i
q = 4096   # (an address that nothing reads)
for B, h, hk, S in ((1, 12, 12, 64), (4, 12, 4, 64), (4, 16, 4, 700), (4, 16, 4, 769)):
    got = go(q, q, q, hk * 800 * 64, 800 * 64, 64, q, q, 1 << 30, B, h, hk, S, S, None, 0.125, None)
    print(int(got != 0) if sys.argv[2] == "taken" else got, end=" ")
"""


def calls(what, **switches):
    """For each call: 1 / 0, taken (and its launch failed) or left to others; or what it returned."""
    from vyomai_amd import _lib
    env = {k: v for k, v in os.environ.items() if not k.startswith("VY_DEC_")}
    out = subprocess.run([sys.executable, "-c", CHILD, _lib.LIB_PATH, what], env={**env, "HIP_VISIBLE_DEVICES": "-1", **switches}, capture_output=True,
                         text=True, timeout=120)
    assert out.returncode == 0, out.stderr[-2000:]
    return [int(v) for v in out.stdout.split()]


no_gpu = pytest.mark.skipif(torch.cuda.device_count() > 0, reason="the addresses are made up: only where no launch succeeds")


@no_gpu
@pytest.mark.parametrize("switches,want", [({}, [1, 1, 0, 0]), ({"VY_DEC_ATTN": "0"}, [0, 0, 0, 0]), ({"VY_DEC_ATTN_NT": "1"}, [0, 0, 0, 0]),
                                           ({"VY_DEC_ATTN_NT": "0"}, [1, 1, 0, 0]), ({"VY_DEC_ATTN_GQ": "0"}, [1, 1, 1, 0])])
def test_switches(switches, want):
    """Four query heads of a key head together stop at 640 keys; each by itself (VY_DEC_ATTN_GQ = 0) at 768, as all contexts do."""
    assert calls("taken", **switches) == want


@no_gpu
def test_a_launch_that_fails_is_an_error():
    assert calls("returned") == [-3, -3, 0, 0]     # VY_ERR_LAUNCH, not a number of shares that nothing wrote
