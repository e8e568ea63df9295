"""The extension a submit goes through (hyle_amd/csrc/submit.cc) passes on what ctypes would: seen from a function of
hyle_hip_plan_launch's signature that notes its arguments.  No GPU."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from hyle_amd import capi

extension = pytest.importorskip("hyle_amd._submit")

SEEN = []


@C.CFUNCTYPE(C.c_int, C.c_void_p, C.POINTER(C.c_void_p), C.c_uint32, C.POINTER(C.c_void_p), C.c_uint32, C.c_void_p, C.c_size_t, C.c_void_p)
def noting(plan, inputs, input_count, outputs, output_count, workspace, size, stream):
    SEEN.append((plan, [inputs[i] for i in range(input_count)], [outputs[i] for i in range(output_count)], workspace, size, stream))
    return 7


NOTING = C.cast(noting, C.c_void_p).value


@pytest.mark.parametrize("inputs,outputs", [([], []), ([1], [2]), ((0x7F0000000000, None), [(1 << 64) - 256]), ([1, 2, 3, 4], (5, 6)),
                                            ([C.c_void_p(9), C.c_void_p(None), 0], [C.c_void_p(8)])])
def test_arguments_arrive(inputs, outputs):
    plain = [[getattr(a, "value", a) or None for a in side] for side in (inputs, outputs)]
    for plan, workspace, size, stream in ((None, 0, 0, 0), (0x1234, 0x7F1200000000, (1 << 40) + 3, C.c_void_p(0x55))):
        SEEN.clear()
        assert extension.launch(NOTING, plan, inputs, outputs, workspace, size, stream) == 7
        assert SEEN == [(plan, *plain, workspace or None, size, getattr(stream, "value", stream) or None)]


def test_what_cannot_be_an_address_is_refused():
    SEEN.clear()
    for inputs, outputs, error in (([1.0], [1], TypeError), (["1"], [1], TypeError), ([np.float32(1)], [1], TypeError), (3, [1], TypeError),
                                   ([1] * (capi.MAX_INPUTS + 1), [1], IndexError), ([1], [1] * (capi.MAX_OUTPUTS + 1), IndexError)):
        with pytest.raises(error):
            extension.launch(NOTING, 1, inputs, outputs, 0, 0, 0)
    with pytest.raises(TypeError):
        extension.launch(NOTING, 1, [1], [1], 0, "8", 0)
    with pytest.raises(TypeError):
        extension.launch(NOTING, 1)
    assert SEEN == []
