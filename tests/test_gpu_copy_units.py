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


@pytest.mark.parametrize("size", list(DTYPES))
def test_copy_units(size):
    rng = np.random.default_rng(1830 + size)
    flat = torch.from_numpy(rng.integers(0, 256, 1 << 21, dtype=np.uint8)).to(DEVICE)
    for offset in (0, 8 if size <= 8 else 0, size, 3 * size):
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
            if name in ("heads in front of tokens", "rows further apart") and size > 1 and offset % 16 == 0:
                assert hc.last_launch_variant() == "copy_units"
