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


TRACE = """
class Builder(rt.ProgramBuilder):    # host tensors of [64, 96] are fp32, their slots bf16
    def input(self, shape, dtype, layout=TL.Tile, storage=ST.Device):
        return super().input(shape, DT.Float32 if storage == ST.Host and tuple(shape) == (64, 96) else dtype, layout, storage)
small = [((33, 70), DT.BFloat16), ((1, 128), DT.Float32), ((17,), DT.Float32, TL.RowMajor), ((5, 7), DT.BFloat16)]
large = [((450, 500 + i), DT.Float32) for i in range(11)]     # 0.9 MB each: more than the staging block holds
args = small + large[:6] + [((3, 40, 33), DT.BFloat16), ((600, 1000), DT.Float32), ((64, 96), DT.BFloat16)] + large[6:] + small + [((2, 40), DT.Float32)]
if ALONE: args = args[:1]
args = [(a[0], a[1], False) + a[2:] for a in args]
def body(pb, ids):
    tiled = [pb.to_layout(i, TL.Tile) if len(a) > 3 else i for a, i in zip(args, ids)]
    return [pb.binary(programs.BINARY["add"], t, t) for t in tiled]
pb = Builder()
emit = programs.add_traced(pb, "sums", args, body, [(a[0], rt.Layout(ST.Device, TL.Tile, a[1])) for a in args])
pb.begin_program("sums")
for y in emit(pb, [pb.input(a[0], a[1], TL.RowMajor, ST.Host) for a in args]):
    pb.output(y)
pb.end_program()
binary = rt.Binary.load_from_memory(pb.finish())
torch_type = {DT.BFloat16: torch.bfloat16, DT.Float32: torch.float32}
def values(step):
    g = torch.Generator().manual_seed(step)
    return [torch.randn(a[0], generator=g).to(torch.float32 if a[0] == (64, 96) else torch_type[a[1]]) for a in args]
def step(tensors):
    return [rt.to_torch(rt.to_host(y, untilize=True)[0]) for y in rt.submit(device, binary, binary.get_num_programs() - 1, tensors)]
def check(got, xs):
    for a, y, x in zip(args, got, xs):
        assert torch.equal(y, x.to(torch_type[a[1]]) * 2), a
"""


def test_host_inputs_of_a_traced_step(null_env):  # noqa: F811
    """More of them than a launch takes and than the staging block holds at once, between them one with a change of type, a batch of matrices
    and one over 1 MiB; then some of them new, none, and a step with one input."""
    run(null_env, "ALONE = False" + TRACE + """
assert len(args) == 23 and sum(a[0][0] * a[0][-1] * 4 for a in args if a[0][0] == 450) > 8 << 20
for s in range(3):
    xs = values(s)
    rt.clear_stats()
    check(step([rt.from_torch(x) for x in xs]), xs)
    assert rt.get_stat("StagingBlockReused") >= 1
kept = [rt.from_torch(x) for x in xs]
check(step(kept), xs)
check(step(kept), xs)
for i in (0, 4, 10, 12, 22):
    xs[i] = values(9)[i]
    kept[i] = rt.from_torch(xs[i])
    check(step(kept), xs)
""")
    run(null_env, "ALONE = True" + TRACE + """
for s in range(3):
    check(step([rt.from_torch(x) for x in values(s)]), values(s))
""")


def test_a_traced_step_that_failed_leaves_no_stale_input(null_env):  # noqa: F811
    """A launch of a step's uploads fails; the step before it, given again, must not find the new values where the failed one had brought them."""
    run(null_env, "ALONE = False" + TRACE + """
import ctypes
null = ctypes.CDLL(os.environ["TTMLIR_AMD_HIP_LIB"])
before = values(1)
kept = [rt.from_torch(x) for x in before]
check(step(kept), before)
check(step(kept), before)
for n in range(1, 40):
    null.ttm_set_option(b"null_device_fail_in", n)
    try:
        step([rt.from_torch(x) for x in values(1 + n)])
    except RuntimeError as e:
        assert "was to fail" in str(e)
    else:
        break
    check(step(kept), before)
assert 5 < n < 39
null.ttm_set_option(b"null_device_fail_in", 0)
check(step(kept), before)
""")
