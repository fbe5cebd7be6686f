"""The phase-trace build's launch ring over ragged calls, whose grids hold
workgroups without a piece: every launch advances it by one."""

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..")

CHILD = """
import ctypes
import numpy as np
import torch
import hyquant_amd as hq
from hyquant_amd import _lib
L = _lib.lib()
L.hyq_phase_trace_geometry.restype = None
s, w, n = (ctypes.c_int32() for _ in range(3))
L.hyq_phase_trace_geometry(ctypes.byref(s), ctypes.byref(w), ctypes.byref(n))
buf = np.zeros(s.value * w.value * n.value, np.uint64)
def launches():
    c = ctypes.c_uint32()
    assert L.hyq_phase_trace_read(buf.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(buf.nbytes), ctypes.byref(c)) == 0
    return c.value
BHK, G, nq, nb = 64, 4, 12000, 64           # shared by all heads: above the line of the device's plan
code = torch.randint(-128, 128, (1, nq, 64), dtype=torch.int8, device="cuda").expand(BHK, -1, -1)
scale = torch.full((1, nq), 0.1, dtype=torch.float16, device="cuda").expand(BHK, -1)
rows = torch.randn(1, nb, 128, device="cuda").bfloat16().expand(BHK, -1, -1)
q = torch.randn(BHK * G, 128, device="cuda").bfloat16()
for share in (0.05, 1.0, 0.3):
    lq = torch.full((BHK,), int(nq * share), dtype=torch.int32, device="cuda")
    lb = torch.full((BHK,), nb, dtype=torch.int32, device="cuda")
    before = launches()
    for _ in range(3):
        hq.fused_d_stage_decode_batched(q, code, code, scale, scale, rows, rows, lq, lb, 4, 4, kv_repeat=G)
    assert launches() == before + 3, (share, before, launches())
print("ok")
"""


def test_ragged_launches_advance_the_trace_ring():
    from hyquant_amd.build import TRACE_LIB
    if not os.path.exists(TRACE_LIB):
        pytest.skip("the phase-trace library is not built (python -m hyquant_amd.build --trace)")
    env = dict(os.environ, HYQ_LIBRARY=TRACE_LIB)
    proc = subprocess.run([sys.executable, "-c", CHILD], cwd=ROOT, env=env, capture_output=True, text=True, timeout=100)
    assert proc.returncode == 0 and "ok" in proc.stdout, proc.stderr[-2000:]
