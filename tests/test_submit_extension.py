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


class Tensor:
    """What launch_tensors asks a tensor for."""

    def __init__(self, address, also=None):
        self.address, self.also = address, also

    def data_ptr(self):
        if self.also is not None:
            self.also()
        return self.address


def test_tensors_arrive_with_the_current_stream_and_what_fails_is_not_launched():
    asked = []

    def stream_of(device):
        asked.append(device)
        return 0x55

    for inputs, outputs in (([], ()), ([Tensor(1), Tensor(0)], (Tensor((1 << 64) - 256),)), ((Tensor(3),) * 4, [Tensor(5), Tensor(6)])):
        SEEN.clear()
        assert extension.launch_tensors(NOTING, lambda: 3, stream_of, 0x1234, inputs, outputs, 0x100, 512) == 7
        assert SEEN == [(0x1234, [t.address or None for t in inputs], [t.address for t in outputs], 0x100, 512, 0x55)]
    assert asked == [3, 3, 3]
    SEEN.clear()
    shrinking = [Tensor(1), Tensor(2)]
    shrinking[0].also = shrinking.clear

    def no_device():
        raise RuntimeError("no device")

    for device, inputs, outputs, size, error in ((lambda: 3, [1], [], 0, AttributeError), (lambda: 3, [Tensor("1")], [], 0, TypeError),
                                                 (lambda: 3, [], iter([]), 0, TypeError), (lambda: 3, [Tensor(1)] * (capi.MAX_INPUTS + 1), [], 0, IndexError),
                                                 (lambda: 3, [], [Tensor(1)] * (capi.MAX_OUTPUTS + 1), 0, IndexError), (lambda: 3, shrinking, [], 0, RuntimeError),
                                                 (no_device, [], [], 0, RuntimeError), (lambda: 3, [], [], "8", TypeError)):
        with pytest.raises(error):
            extension.launch_tensors(NOTING, device, stream_of, 1, inputs, outputs, 0, size)
    assert SEEN == []
