"""Copy of strided tensors in units of 2 to 16 bytes (cast.hip, copy_units): every unit, folded and
unfolded axes, broadcast axes, odd strides and addresses that leave it.  The bytes stay the same."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from hyle_amd import compute as hc

from gpu_support import DEVICE, note, run

pytestmark = pytest.mark.gpu

DTYPES = {1: torch.uint8, 2: torch.int16, 4: torch.int32, 8: torch.int64}


def widest_unit(shape, strides, size, address):
    """The most bytes, up to 16, that the copy can move at once: a power of two such that every run of that many bytes of
    the result comes from one place that is a multiple of it (1: no run of two bytes does)."""
    at = sum(np.arange(n).reshape([-1] + [1] * (len(shape) - 1 - axis)) * (step * size)
             for axis, (n, step) in enumerate(zip(shape, strides))) + np.zeros(shape, np.int64) + address
    at = at.reshape(-1)
    unit = 16
    while unit > size:
        many = unit // size
        if at.size % many == 0:
            runs = at.reshape(-1, many)
            if np.all(runs[:, 0] % unit == 0) and np.array_equal(runs, runs[:, :1] + np.arange(many) * size):
                return unit
        unit //= 2
    return size


@pytest.mark.parametrize("size", list(DTYPES))
def test_copy_units(size):
    rng = np.random.default_rng(1830 + size)
    seen = set()
    flat = torch.from_numpy(rng.integers(0, 256, 1 << 21, dtype=np.uint8)).to(DEVICE)
    for offset in sorted({0, 2, 4, 8, size, 3 * size} - {n for n in (2, 4) if n % size != 0}):
        base = flat[offset:offset + (((1 << 21) - 64) // size) * size].view(DTYPES[size])
        for name, shape, strides in (
                ("heads in front of tokens", (5, 33, 64), (64, 320, 1)), ("a run of eight bytes' worth", (7, 9, 8), (8, 64, 1)),
                ("an odd run", (6, 11, 13), (13, 90, 1)), ("a plain transpose", (129, 65), (1, 129)), ("rows further apart", (37, 48), (64, 1)),
                ("a broadcast axis", (4, 6, 32), (32, 0, 1)), ("a broadcast last axis", (50, 6), (2, 0)), ("folded outer axes", (3, 4, 5, 16), (640, 160, 32, 1)),
                ("five axes", (3, 2, 5, 4, 8), (8, 24, 192, 48, 1)), ("every second", (1, 300), (7, 2)), ("one element", (1, 1), (3, 5))):
            view = base.as_strided(shape, strides)
            note(f"copy units of {size}-byte elements, {offset} bytes off: {name}")
            (out,) = run(hc.Copy(), view)
            assert torch.equal(out, view.contiguous()), (size, offset, name)
            if not view.is_contiguous() and view.numel() > 1:
                unit = widest_unit(shape, strides, size, view.data_ptr())
                label = f"copy_units/{unit}" if unit >= max(2, size) else "cast_general"
                assert hc.last_launch_variant().startswith(label), (size, offset, name, label, hc.last_launch_variant())
                seen.add(unit)
    assert seen == {unit for unit in (1, 2, 4, 8, 16) if unit >= size}   # every unit that this element size can have
