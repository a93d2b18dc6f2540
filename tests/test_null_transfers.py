"""Host <-> device transfers of the runtime on the null device (tests/cpp/null_device.cpp), whose page-locked memory the kernels reach
as on the GPU: what is staged, what waits, and the values that arrive."""
import os
import subprocess
import sys

import pytest

from test_null_device import null_env  # noqa: F401 (fixture)

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SETUP = """
import sys, os
sys.path.insert(0, %r)
import __graft_entry__ as entry
entry.load_package()
import torch
from ttmlir_amd import datagen, programs, runtime as rt
DT, TL, ST = rt.DataType, rt.TensorLayout, rt.StorageType
device = rt.open_mesh_device()
""" % ROOT


def run(env, code, timeout=120):
    r = subprocess.run([sys.executable, "-c", SETUP + code], env=env, capture_output=True, text=True, timeout=timeout, cwd=ROOT)
    assert r.returncode == 0, r.stdout[-500:] + r.stderr[-1500:]
    return r.stdout


def test_an_upload_is_staged_once(null_env):  # noqa: F811
    """Eight tensors of 2 MiB through the 8 MiB block, with changes of type that no single kernel makes on the way: it is used up once."""
    run(null_env, """
xs = [datagen.randn((512, 1024), seed=i) for i in range(8)]
rt.clear_stats()
ds = [rt.to_layout(rt.from_torch(x), device, rt.Layout(ST.Device, TL.Tile, DT.BFloat16)) for x in xs]
assert rt.get_stat("StagingBlockReused") == 1, rt.get_stat("StagingBlockReused")
for x, d in zip(xs, ds):
    assert torch.equal(rt.to_torch(d), x.to(torch.bfloat16))
""")


def test_uploads_are_waited_for_beside_another_open_handle(null_env):  # noqa: F811
    """Every handle has a stream of its own and the device pool is common: a tensor that is still on its way on one stream could be
    read, or its memory reused, on the other."""
    run(null_env, """
import ctypes
null = ctypes.CDLL(os.environ["TTMLIR_AMD_HIP_LIB"])
null.null_device_syncs.restype = ctypes.c_long
def waits(f):
    before = null.null_device_syncs()
    f()
    return null.null_device_syncs() - before
plain, tiled = rt.Layout(ST.Device, TL.RowMajor, DT.Float32), rt.Layout(ST.Device, TL.Tile, DT.Float32)
x = torch.randn(64, 96)
up = lambda d, lay: rt.to_layout(rt.from_torch(x), d, lay)
assert waits(lambda: up(device, plain)) == waits(lambda: up(device, tiled)) == 0
others = []
assert waits(lambda: others.append(rt.open_mesh_device())) >= 2      # its own probe, and what the first handle has under way
for d in (device, others[0]):
    assert waits(lambda: up(d, plain)) == waits(lambda: up(d, tiled)) == 1
rt.close_mesh_device(others[0])
assert waits(lambda: up(device, plain)) == waits(lambda: up(device, tiled)) == 0
""")
