"""Bound.submit without a stream asks for the current stream and the tensors' addresses natively (launch_tensors of
hyle_amd/csrc/submit.cc): from the first submit on, on whatever stream is current, under capture, and with what the library
refuses.  OperationInvocation.submit is taken out of the way, so that no other path can answer."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from hyle_amd import capi
from hyle_amd import compute as hc
from hyle_amd import torch_io as tio
from oracle import lib as orc

from gpu_support import DEVICE, assert_bits_equal, assert_close_f32, context, note, to_device, to_host

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def native_only(monkeypatch):
    context()
    torch.empty(1, device=DEVICE)   # torch has initialised the device
    if tio._raw_stream is None or capi.launcher() is capi.launch_through_ctypes:
        pytest.skip("the extension was not built, or torch offers no bare stream handle")

    def elsewhere(self, *args):
        raise AssertionError("this submit did not go through launch_tensors")
    monkeypatch.setattr(hc.OperationInvocation, "submit", elsewhere)


def norm_and_topk(rng):
    """An operation of two inputs, and one with two outputs and a workspace, with what the oracle says."""
    x, w = rng.normal(0, 1, (37, 1000)).astype(np.float32), rng.normal(1, 0.1, 1000).astype(np.float32)
    logits = rng.permutation(3 * 40000).reshape(3, 40000).astype(np.float32)
    want = (orc.rms_norm(orc.F32, x, w, 1e-6, weight_type=orc.F32), -np.sort(-logits, 1)[:, :16], np.argsort(-logits, 1, kind="stable")[:, :16])
    return [to_device(x, "f32"), to_device(w, "f32")], [to_device(logits, "f32")], want


def hold(norm_outs, topk_outs, want):
    assert_close_f32(to_host(norm_outs[0]), want[0], rel=1e-5)
    assert np.array_equal(to_host(topk_outs[0]), want[1]) and np.array_equal(to_host(topk_outs[1]), want[2])


def bounds_for(norm_inputs, topk_inputs):
    return (tio.Bound(context(), hc.RmsNorm(1e-6), [tio.desc_of(t) for t in norm_inputs]),
            tio.Bound(context(), hc.TopK(count=16), [tio.desc_of(t) for t in topk_inputs]))


def test_first_and_later_submits_with_other_buffers_lists_and_tuples():
    norm, topk = None, None
    for seed in range(3):
        norm_inputs, topk_inputs, want = norm_and_topk(np.random.default_rng(1900 + seed))
        if norm is None:
            norm, topk = bounds_for(norm_inputs, topk_inputs)
        outs = norm.outputs(), topk.outputs()
        note(f"native submit, pass {seed}")
        norm.submit(tuple(norm_inputs) if seed == 1 else norm_inputs, outs[0])
        topk.submit(topk_inputs, tuple(outs[1]) if seed == 1 else outs[1])
        torch.cuda.synchronize()
        hold(*outs, want)


def test_the_current_stream_is_the_one_taken():
    norm_inputs, topk_inputs, want = norm_and_topk(np.random.default_rng(1910))
    norm, topk = bounds_for(norm_inputs, topk_inputs)
    side = torch.cuda.Stream()
    outs = norm.outputs(), topk.outputs()
    late = torch.zeros_like(norm_inputs[0])
    norm.submit([late, norm_inputs[1]], outs[0])   # the kernels are loaded
    topk.submit(topk_inputs, outs[1])
    for t in (*outs[0], *outs[1]):
        t.zero_()
    side.wait_stream(torch.cuda.current_stream())
    note("native submit on a side stream, behind a copy that only this stream orders before it")
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)              # some ten milliseconds
        late.copy_(norm_inputs[0])
        norm.submit([late, norm_inputs[1]], outs[0])
        topk.submit(topk_inputs, outs[1])
    side.synchronize()                             # (a launch on another stream read zeros)
    hold(*outs, want)


def test_capture_without_a_stream_of_the_caller_s():
    norm_inputs, topk_inputs, want = norm_and_topk(np.random.default_rng(1920))
    norm, topk = bounds_for(norm_inputs, topk_inputs)
    outs = norm.outputs(), topk.outputs()
    note("native submit: eager pass before the capture")
    norm.submit(norm_inputs, outs[0])
    topk.submit(topk_inputs, outs[1])
    torch.cuda.synchronize()
    eager = [to_host(t).copy() for t in (*outs[0], *outs[1])]
    hold(*outs, want)
    graph = torch.cuda.CUDAGraph()
    note("native submit: capture")
    with torch.cuda.graph(graph):
        norm.submit(norm_inputs, outs[0])
        topk.submit(topk_inputs, outs[1])
    for replay in range(3):
        for t in (*outs[0], *outs[1]):
            t.zero_()
        topk.workspace.fill_(0xFF if replay % 2 else 0)
        torch.cuda.synchronize()
        note(f"native submit: replay {replay}")
        graph.replay()
        torch.cuda.synchronize()
        for got, expected in zip((*outs[0], *outs[1]), eager):
            assert_bits_equal(to_host(got).view(np.uint32), expected.view(np.uint32))


def test_what_the_library_refuses_is_raised_and_not_launched():
    norm_inputs, topk_inputs, want = norm_and_topk(np.random.default_rng(1930))
    norm, topk = bounds_for(norm_inputs, topk_inputs)
    outs = norm.outputs(), topk.outputs()
    outs[0][0].fill_(7.0)
    empty = torch.empty(0, device=DEVICE)    # its address is null
    for inputs, outputs in ((norm_inputs[:1], outs[0]), (norm_inputs, []), (norm_inputs * 2, outs[0]), ([norm_inputs[0], empty], outs[0]),
                            (norm_inputs, [empty])):
        note("native submit with bindings that the library refuses")
        with pytest.raises(hc.StatusError):
            norm.submit(inputs, outputs)
    with pytest.raises(IndexError):
        norm.submit(norm_inputs * capi.MAX_INPUTS, outs[0])
    with pytest.raises(AttributeError):
        norm.submit([norm_inputs[0], 5], outs[0])
    torch.cuda.synchronize()
    assert (outs[0][0] == 7.0).all()
    norm.submit(norm_inputs, outs[0])        # and the next one is an ordinary one
    topk.submit(topk_inputs, outs[1])
    torch.cuda.synchronize()
    hold(*outs, want)
