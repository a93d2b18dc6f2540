"""Options that pin a launch plan of the linear kernels: a plan that does not exist is an error return, on the host, before any launch."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CODE = r"""
import ctypes, sys
sys.path.insert(0, %r)
import __graft_entry__ as entry
entry.load_package()
from ttmlir_amd import hip
l, I64 = hip.lib(), ctypes.c_int64
l.ttm_set_option(b"check_extents", 0)     # the operands below are addresses nothing may follow
l.ttm_set_option(b"linear_mid", %d)
p = lambda i: ctypes.c_void_p(4096 * (i + 1))
if %d:
    rc = l.ttm_linear_glu(p(0), p(1), p(2), hip.BFP8B, p(3), I64(65), I64(5760), I64(512), 2, 0, None)
else:
    rc = l.ttm_linear(p(0), hip.BF16, p(1), hip.BFP8B, 0, None, hip.BF16, hip.TILE, p(3), hip.BF16, I64(1), I64(1), I64(96), I64(512), I64(512), 0, None)
print(rc, l.ttm_last_error().decode())
"""


@pytest.mark.parametrize("plan,gated", [(4401, 0), (8301, 0), (8103, 0), (1000, 0), (8101, 1), (8201, 1), (4202, 1)])
def test_a_pinned_plan_that_does_not_exist_is_refused(plan, gated):
    r = subprocess.run([sys.executable, "-c", CODE % (ROOT, plan, gated)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-400:]
    assert r.stdout.startswith("1 ") and "no such plan" in r.stdout and str(plan) in r.stdout
