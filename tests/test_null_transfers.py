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


def test_reading_a_tensor_of_a_busy_handle_does_not_wait_for_its_program(null_env):  # noqa: F811
    """A thread that holds one handle's lock (to_layout on it) and reads a tensor of another, whose program waits for that thread."""
    run(null_env, """
import threading
other = rt.open_mesh_device()
x = torch.randn(64, 96)
mine = rt.to_layout(rt.from_torch(x), device, rt.Layout(ST.Device, TL.Tile, DT.Float32), retain=True)
got = []
def reader():
    got.append(rt.to_torch(rt.to_layout(mine, other, rt.Layout(ST.Host, TL.RowMajor, DT.Float32))))
def hook(idx, name, dbg, h):
    if not got and not threads:
        threads.append(threading.Thread(target=reader, daemon=True))
        threads[0].start()
        threads[0].join(30)
        finished.append(not threads[0].is_alive())
        if not finished[0]:
            os._exit(3)
threads, finished = [], []
rt.set_post_op_callback(hook)
b = rt.Binary.load_from_memory(programs.c1_matmul())
ins = [rt.to_layout(rt.from_torch(t), device, rt.get_layout(b, 0, i)) for i, t in enumerate(datagen.c1_matmul())]
rt.submit(device, b, 0, ins)
assert finished == [True] and torch.equal(got[0], x)
""")


def test_a_callback_after_the_program_sees_every_result_as_declared(null_env):  # noqa: F811
    """Layout changes that are made on the way over PCIe leave their operand in the result's place: not where a callback may read the
    result (wrong layout and type) or write it (into the caller's input)."""
    run(null_env, """
pb = rt.ProgramBuilder()
pb.begin_program("p")
a = pb.input((64, 96), DT.Float32, TL.RowMajor, ST.Host)
up = pb.to_device(a)
t = pb.to_layout(up, TL.Tile)
s = pb.unary(programs.UNARY["neg"], t)
down = pb.to_layout(s, TL.RowMajor, DT.BFloat16)
out = pb.from_device(down)
pb.output(out)
pb.end_program()
b = rt.Binary.load_from_memory(pb.finish())
x = torch.randn(64, 96)
host = rt.from_torch(x)
seen = {}
def post(idx, hook):
    seen["down"] = hook.retrieve(down, untilize=False).desc()[1]
    seen["up"] = rt.to_torch(hook.retrieve(up))
    hook.update(up, rt.from_torch(torch.zeros(64, 96)))
rt.set_program_callbacks(post=post)
(y,) = rt.submit(device, b, 0, [host])
assert (seen["down"].layout, seen["down"].dtype) == (TL.RowMajor, DT.BFloat16)
assert torch.equal(seen["up"], x) and torch.equal(rt.to_torch(host), x)
assert torch.equal(rt.to_torch(y), -x.to(torch.bfloat16))
""")


def test_a_round_trip_through_the_device_is_a_copy(null_env):  # noqa: F811
    """to_device, then a to_layout back to the host that changes nothing: the result is not the caller's tensor."""
    run(null_env, """
pb = rt.ProgramBuilder()
pb.begin_program("p")
a = pb.input((64, 96), DT.Float32, TL.RowMajor, ST.Host)
pb.output(pb.to_layout(pb.to_device(a), TL.RowMajor, DT.Float32, ST.Host))
pb.end_program()
x = torch.randn(64, 96)
host = rt.from_torch(x)
(y,) = rt.submit(device, rt.Binary.load_from_memory(pb.finish()), 0, [host])
assert rt.host_data_ptr(y) != rt.host_data_ptr(host)
rt.memcpy_tensor(host, rt.from_torch(torch.zeros(64, 96)))
assert torch.equal(rt.to_torch(y), x)
""")


@pytest.mark.parametrize("pageable", ["0", "1"])
def test_transfers_on_both_routes(null_env, pageable):  # noqa: F811
    """The GPU's transfer tests, with page-locked memory within the kernels' reach and without (the memcpy routes)."""
    skip = "not through_page_locked" if pageable == "1" else ""
    r = subprocess.run([sys.executable, "-m", "pytest", os.path.join(ROOT, "tests", "test_gpu_transfers.py"), "-q", "-m", "gpu", "-p", "no:cacheprovider",
                        "-k", skip], env=dict(null_env, TTMLIR_AMD_NULL_DEVICE_PAGEABLE=pageable), capture_output=True, text=True, timeout=600, cwd=ROOT)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-1000:]
