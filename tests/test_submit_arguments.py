"""OperationInvocation.submit takes and refuses what ctypes does, with the extension of hyle_amd/csrc/submit.cc and
without it: seen from a function of hyle_hip_plan_launch's signature that notes its arguments.  No GPU."""
from __future__ import annotations

import ctypes as C
import functools
import os
import sys
import sysconfig
from types import SimpleNamespace

import numpy as np
import pytest

from hyle_amd import capi
from hyle_amd import compute as hc

SEEN = []


@C.CFUNCTYPE(C.c_int, C.c_void_p, C.POINTER(C.c_void_p), C.c_uint32, C.POINTER(C.c_void_p), C.c_uint32, C.c_void_p, C.c_size_t, C.c_void_p)
def noting(plan, inputs, input_count, outputs, output_count, workspace, size, stream):
    SEEN.append((plan, [inputs[i] for i in range(input_count)], [outputs[i] for i in range(output_count)], workspace, size, stream))
    return capi.OK


class StreamObject:
    """What torch's stream objects are to ctypes."""
    _as_parameter_ = C.c_void_p(0x77)


@pytest.fixture(params=["extension", "ctypes"])
def invocation(request, monkeypatch):
    library = SimpleNamespace(hyle_hip_plan_launch=noting, hyle_hip_last_launch_variant=lambda: b"")   # the GPU tests ask for the label
    monkeypatch.setattr(capi, "load", lambda: library)
    if request.param == "ctypes":                                      # as if it had not been built
        monkeypatch.setitem(sys.modules, "hyle_amd._submit", None)
        monkeypatch.delattr("hyle_amd._submit", raising=False)
        monkeypatch.setattr(os.path, "exists", lambda path: False)
    elif not os.path.exists(os.path.join(sysconfig.get_paths()["include"], "Python.h")):
        pytest.skip("no Python headers: the extension is not built")
    launch = capi.launcher.__wrapped__()
    assert isinstance(launch, functools.partial) == (request.param == "extension")
    made = object.__new__(hc.OperationInvocation)
    made._prepared, made._workspace, made._workspace_size, made._launch = SimpleNamespace(_handle=0x1234), 0x100, 512, launch
    SEEN.clear()
    return made


@pytest.mark.parametrize("stream,handle", [(0, None), (0x77, 0x77), (None, None), (C.c_void_p(0x77), 0x77), (StreamObject(), 0x77)])
def test_streams(invocation, stream, handle):
    invocation.submit(stream, (0x10, C.c_void_p(0x20)), [0x30])
    assert SEEN == [(0x1234, [0x10, 0x20], [0x30], 0x100, 512, handle)]


def test_sequences(invocation):
    for inputs in ([], (1, 2, 3, 4), {7: "a", 8: "b"}.keys(), range(2, 4), [None, True]):
        SEEN.clear()
        invocation.submit(0, inputs, (5, 6))
        assert SEEN == [(0x1234, [int(i) if i else None for i in inputs], [5, 6], 0x100, 512, None)]


@pytest.mark.parametrize("inputs", [[C.c_int(3)], [C.c_uint64(3)], [SimpleNamespace(value=3)], [StreamObject()], ["3"], [b"3"], [1.0], [np.int64(3)],
                                    iter([3]), 3])
def test_what_is_no_address(invocation, inputs):
    with pytest.raises(TypeError):
        invocation.submit(0, inputs, [0x30])
    with pytest.raises(TypeError):
        invocation.submit(0, [0x10], inputs)
    assert SEEN == []


@pytest.mark.parametrize("stream", [C.c_int(3), SimpleNamespace(value=3), 1.5])
def test_what_is_no_stream(invocation, stream):
    with pytest.raises(C.ArgumentError):
        invocation.submit(stream, [0x10], [0x30])
    assert SEEN == []


def test_too_many(invocation):
    with pytest.raises(IndexError):
        invocation.submit(0, [1] * (capi.MAX_INPUTS + 1), [0x30])
    with pytest.raises(IndexError):
        invocation.submit(0, [1], [0x30] * (capi.MAX_OUTPUTS + 1))
    assert SEEN == []
