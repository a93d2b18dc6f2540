"""call() and ptr() as compiled code (binding/py_call.cpp) against the ctypes functions they stand for: the same conversions, the same
errors.  What an argument arrived as shows in the entry points' own messages; nothing is launched."""
import ctypes
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest
import torch


def outcome(fn, *args):
    try:
        return fn(*args)
    except Exception as e:
        return type(e), str(e)


def activation(hip, call, value, p=16):
    return outcome(call, "ttm_linear", p, hip.BF16, p, hip.BFP8B, 0, None, hip.BF16, hip.TILE, p, hip.BF16, 1, 1, 32, 32, 32, value, None)


@pytest.fixture(autouse=True)
def unchecked(hip):
    was_on = hip._check_buffers
    hip.check_buffers(False)   # the messages under test are those of arguments that the size check would stop
    yield
    hip.check_buffers(was_on)


@pytest.mark.parametrize("value", [9, -1, True + 8, 2 ** 32 + 7, 2 ** 64 + 5, -(2 ** 63) - 6, np.int64(9), np.int32(-3), 1.5, "x", None, ctypes.c_int(9)])
def test_integers(hip, value):
    got = activation(hip, hip.call, value)
    assert got == activation(hip, hip._call, value) and got is not None


@pytest.mark.parametrize("dst", [None, 0, 3, 2 ** 64 + 3, ctypes.c_void_p(), ctypes.c_void_p(3), "address", np.uint64(3), 1.0])
def test_pointers(hip, dst):
    dst = hip._Ptr(3) if isinstance(dst, str) else dst
    got = outcome(hip.call, "ttm_fill_u32", dst, 0, 4, None)
    assert got == outcome(hip._call, "ttm_fill_u32", dst, 0, 4, None) and got is not None


def test_other_arguments_go_through_ctypes(hip):
    v = ctypes.c_int(0)
    hip.call("ttm_set_option", b"linear_mid", 7)
    hip.call("ttm_get_option", b"linear_mid", ctypes.byref(v))
    hip.call("ttm_set_option", b"linear_mid", 0)
    assert v.value == 7
    for args in (("ttm_fill_u32", None, 0), ("no_such_entry",), ("ttm_clamp", 16, 16, 0, 0, 1, 1, 1, "a", 0.0, None), ()):
        got = outcome(hip.call, *args)
        assert isinstance(got, tuple) and got[0] == outcome(hip._call, *args)[0], args


def test_every_status_function_is_bound(hip):
    bound = set(hip._native.names())
    for name, res, argtypes in hip.declared_functions():
        plain = res is ctypes.c_int and ctypes.c_char_p not in argtypes and name != "ttm_device_name"
        assert (name in bound) == plain, name


def test_floats(hip):
    # a NULL tensor is refused after the arguments are converted: what is compared is that every kind of number is taken
    for lo in (0.5, 1, True, 2 ** 70, float("nan")):
        args = ("ttm_clamp", None, None, 0, 0, 1, 1, 1, lo, 0.0, None)
        assert outcome(hip.call, *args) == outcome(hip._call, *args)


def test_ptr(hip):
    for t in (torch.zeros(5, 7), torch.zeros(0), torch.zeros(3, dtype=torch.bfloat16)[1:]):
        a, b = hip.ptr(t), hip._ptr(t)
        assert type(a) is type(b) and a.value == b.value and a.nbytes == b.nbytes == t.nbytes
    assert outcome(hip.ptr, torch.zeros(4, 4).t()) == outcome(hip._ptr, torch.zeros(4, 4).t())
    assert outcome(hip.ptr, 5)[0] is AttributeError
    assert hip.ptr(t=t).value == t.data_ptr() and outcome(hip.ptr)[0] is TypeError and outcome(hip.ptr, t, t)[0] is TypeError


def test_keywords(hip):
    assert outcome(lambda: hip.call(name="ttm_fill_u32"))[0] == outcome(lambda: hip._call(name="ttm_fill_u32"))[0]
    assert outcome(lambda: hip.call("ttm_fill_u32", None, 0, 4, stream=None))[0] is TypeError


@pytest.mark.parametrize("built", [False, True])
def test_a_binding_built_after_the_import(hip, tmp_path, built):
    """A process that imports the module, then builds, then calls: it uses the binding that is there by the first call, and without one makes its
    calls through ctypes, with the check of extents."""
    lib = tmp_path / "tt-mlir_amd" / "lib"
    lib.mkdir(parents=True)
    shutil.copy(os.path.join(hip._HERE, "hip.py"), lib.parent)
    os.symlink(os.path.join(hip.ROOT, "include"), tmp_path / "include")
    for f in os.listdir(os.path.dirname(hip.LIB_PATH)):
        if not f.startswith("_ttm_call"):
            os.symlink(os.path.join(os.path.dirname(hip.LIB_PATH), f), lib / f)
    code = """
import shutil, sys, torch
sys.path.insert(0, %r)
import hip
assert hip._native is None
if %r:
    shutil.copy(%r, hip.CALL_PATH)
hip.lib()
assert (hip._native is not None) == %r and (type(hip.call) is type(len)) == %r
t = torch.zeros(16)
for on in (False, True):
    hip.check_buffers(on)
    try:
        hip.call("ttm_tilize", hip.ptr(t), hip.ptr(t), 1, 32, 32, 4 if on else 3, None)
    except hip.TTMError as e:
        print(e)
    else:
        raise SystemExit("accepted")
""" % (str(lib.parent), built, hip.CALL_PATH, built, built)
    done = subprocess.run([sys.executable, "-c", code], env={**os.environ, "TTMLIR_AMD_CHECK_BUFFERS": "0"}, capture_output=True, text=True)
    assert done.returncode == 0, done.stderr
    assert "elem_bytes" in done.stdout and "row-major input" in done.stdout


def test_the_binding_is_one_for_this_python(hip):
    import sysconfig
    assert hip.CALL_PATH.endswith(sysconfig.get_config_var("EXT_SUFFIX")) and type(hip.call) is type(len)


def test_sizes_are_checked_before_the_call(hip):
    hip.check_buffers(True)
    t = torch.zeros(16)
    got = outcome(hip.call, "ttm_tilize", hip.ptr(t), hip.ptr(t), 1, 32, 32, 4, None)
    assert got[0] is hip.TTMError and "row-major input" in got[1]
