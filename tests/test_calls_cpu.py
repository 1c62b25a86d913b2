"""The extension module that Python's calls go through (csrc/python/calls.cpp): what arrays own, and what operator calls refuse."""
import ctypes
import gc
import os
import subprocess
import sys

import numpy as np
import pytest

from tsplit_amd import _calls, gpu_links as L, ndarray as nd
from tsplit_amd._base import LIB_PATH, _LIB


def test_arrays_own_their_memory_and_views_keep_their_parent():
    a = nd.array(np.arange(12, dtype=np.float32).reshape(3, 4), nd.cpu(0))
    assert a.shape == (3, 4) and a.handle is a.handle and a.data_ptr == a.handle.contents.data and a.ctx.device_type == 1
    v = nd.view(a, (12,))
    assert v._owner is a
    a.split_tensor(3)                            # the array lists views that refer to it: a cycle
    assert [p.asnumpy()[0, 0] for p in a.sTensor] == [0, 4, 8] and a.split_number == 3 and a.splitted
    del a
    gc.collect()
    np.testing.assert_array_equal(v.asnumpy(), np.arange(12))
    for shape in ((), (0, 3), [2, np.int64(5)], (1,) * 20):
        assert nd.empty(shape).shape == tuple(int(s) for s in shape)


def test_an_array_lives_through_assigned_attributes_and_a_raw_handle():
    h = nd.DLArrayHandle()
    shape = (ctypes.c_int64 * 2)(2, 3)
    assert _LIB.DLArrayAlloc(shape, ctypes.c_int64(2), nd.cpu(0), ctypes.byref(h), ctypes.c_int(1)) == 0
    a = nd.NDArray(h)
    assert a.handle is h and a.shape == (2, 3) and (a.swap, a.in_gpu, a._keeper) == (False, True, None)
    a.to_swap()
    a.in_gpu = False
    assert a.swap is True and a.in_gpu is False and a._events == {}


def test_calls_refuse_what_they_cannot_take():
    a = nd.empty((2, 3))
    for bad in (None, 3, "x", np.zeros((2, 3), np.float32)):
        with pytest.raises(AssertionError):
            L.relu(a, bad)
    with pytest.raises(RuntimeError):
        L.matrix_multiply(a, False, a, False, a)            # shapes do not conform: refused before any launch
    with pytest.raises(TypeError):
        L.CuDNN_max_pooling2d(a, 2.5, 2, a)
    with pytest.raises(TypeError):
        _calls.DLGpuRelu(a, a)
    with pytest.raises(ValueError):
        nd.empty("ab")
    with pytest.raises(TypeError):
        nd.empty((2, 3), 5)


def test_an_array_of_a_collected_cycle_goes_to_its_recordings_keeper_first():
    """The keeper lies in the same cycle, older than the array: what it holds must not have been cleared when it is asked."""
    from tsplit_amd.stream import _Keeper
    took, h = [], nd.DLArrayHandle()

    class Keeper(_Keeper):
        def take(self, handle, rule):
            took.append((super().take(handle, rule), ctypes.addressof(handle.contents)))
            return took[-1][0]
    keeper, ring = Keeper(), []
    assert _LIB.DLArrayAlloc((ctypes.c_int64 * 1)(4), ctypes.c_int64(1), nd.cpu(0), ctypes.byref(h), ctypes.c_int(1)) == 0
    h.contents.ctx.device_type = 2              # as an array on the device: only those are the keeper's
    a = nd.NDArray(h)
    a._keeper, a._owner = keeper, ring
    ring.extend([keeper, a])
    address = ctypes.addressof(h.contents)
    del a, keeper, ring, h
    gc.collect()
    assert took == [(True, address)]
    h = ctypes.cast(address, nd.DLArrayHandle)
    h.contents.ctx.device_type = 1
    assert _LIB.DLArrayFree(h, ctypes.c_int(1)) == 0


def test_a_library_without_an_operator_is_loaded_and_misses_that_call_alone(tmp_path):
    names = [line.split()[-1] for line in subprocess.run(["nm", "-D", "--defined-only", LIB_PATH], capture_output=True, text=True, check=True).stdout.splitlines()
             if " T " in line and not line.split()[-1].startswith("_")]
    assert "DLGpuTanh" in names and "TSplit_BatchNormReluAdd" in names
    src, lib = tmp_path / "other.c", str(tmp_path / "other.so")
    src.write_text("".join("int %s() { return 0; }\n" % name for name in names if name != "TSplit_BatchNormReluAdd"))
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", lib], check=True)
    program = """
from tsplit_amd import gpu_links as L, ndarray as nd
a = nd.NDArray(None)
L.tanh(a, a)
try:
    L.batch_norm_relu_add(a, a, a, a, a, a, a)
except AttributeError as e:
    print("without", "TSplit_BatchNormReluAdd" in str(e))
"""
    done = subprocess.run([sys.executable, "-c", program], env=dict(os.environ, TSPLIT_LIB_PATH=lib), capture_output=True, text=True,
                          cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert done.stdout.strip() == "without True", done.stderr


def test_eight_bytes_are_no_pointer_and_no_context():
    a, eight = nd.empty((2, 3)), np.zeros(1)
    assert eight.nbytes == ctypes.sizeof(nd.DLContext) == ctypes.sizeof(ctypes.c_void_p)
    for bad in (eight, b"12345678", ctypes.c_double(1)):
        with pytest.raises(TypeError):
            nd.NDArray(bad)
        with pytest.raises(TypeError):
            nd.empty((2, 3), bad)
        with pytest.raises(TypeError):
            a.handle = bad
    stream = type("Stream", (), {"handle": eight})()
    with pytest.raises(TypeError):
        L.relu(a, a, stream)
    assert a.shape == (2, 3)


def test_flags_of_an_array_take_any_truth_value():
    a = nd.empty((2, 3))
    for value in (0, 1, None, "", "yes"):
        a.auto_deleted = value
        assert bool(a.auto_deleted) == bool(value)


def test_a_memory_rule_that_is_no_number_is_refused(monkeypatch):
    a = nd.empty((2, 3))
    monkeypatch.setattr(nd, "MEMORY_MANAGE_RULE", "pool")
    with pytest.raises(TypeError):
        nd.empty((2, 3))
    monkeypatch.undo()
    assert nd.empty((2, 3)).shape == a.shape


def test_the_module_is_of_this_python():
    """Named by its ABI: another Python finds no module, and not one that does not fit it."""
    import sysconfig

    from tsplit_amd import build
    assert _calls.__file__ == build.CALLS and _calls.__file__.endswith(sysconfig.get_config_var("EXT_SUFFIX"))
    assert not os.path.exists(os.path.join(os.path.dirname(build.CALLS), "_calls.so"))


def test_a_pointer_may_be_filled_in_after_the_array_was_made():
    h = nd.DLArrayHandle()
    a = nd.NDArray(h)
    with pytest.raises(AttributeError):
        a.shape
    assert _LIB.DLArrayAlloc((ctypes.c_int64 * 2)(2, 3), ctypes.c_int64(2), nd.cpu(0), ctypes.byref(h), ctypes.c_int(1)) == 0
    assert a.shape == (2, 3) and a.data_ptr == h.contents.data


def test_a_profiler_may_have_fields_of_its_own():
    from tsplit_amd.profiler import Profiler

    class Longer(Profiler):
        _fields_ = [("calls", ctypes.c_int)]
    a = nd.empty((2, 3))
    with pytest.raises(RuntimeError):                       # taken: the shapes do not conform, which the library refuses
        L.matrix_multiply(a, False, a, False, a, profiler=Longer())
    with pytest.raises(TypeError):
        L.matrix_multiply(a, False, a, False, a, profiler=bytearray(ctypes.sizeof(Profiler)))
