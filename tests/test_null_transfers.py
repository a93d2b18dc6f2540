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
