"""Every launch shape of the RMSNorm / LayerNorm kernels is reached by a case here and checked
against the CPU oracle.

Which kernel serves a norm depends on the row width and on the number of rows: widths that a lane
group holds in whole vectors have launch shapes that cover the tensor exactly when the row count is
a multiple of the rows a block takes (norm_exact.h, from 10 MiB on, and for LayerNorm the exact forms of norm.hip);
rows of 65 to 768 vectors take a wave each (norm_tail.h), other widths and row counts the masked shapes of norm.hip, and
widths that are no whole number of 16-byte vectors the generic kernel.  CASES is the table (operator, type, rows, width) ->
label of the launch shape the library must choose; `hyle_hip_last_launch_variant` reports the
shape actually launched.  The last test fails when a norm shape compiled into the library
(`hyle_hip_variant_label`) is reached by no case.

Semantics: src/compute_provider_native/normalization.cc:41-80 (RMSNorm),
src/simd/math/activations.cc:124-175 (LayerNorm); bars as in test_gpu_parity.py and
test_gpu_layer_norm.py.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from hyle_amd import compute as hc
from oracle import lib as orc

from gpu_support import TYPES, assert_close_f32, assert_narrow_ulp, host_values, note, run, to_device, to_host
from test_gpu_layer_norm import layer_bar

pytestmark = pytest.mark.gpu

# (operator, type, rows, width, label)
CASES = [
    ("layer", "f32", 32, 32, "norm_rows/layer/8x1/256/1/exact"),
    ("layer", "f32", 3, 20, "norm_rows/layer/8x1/256/1/ragged"),
    ("layer", "f32", 16, 64, "norm_rows/layer/16x1/256/1/exact"),
    ("layer", "f32", 3, 52, "norm_rows/layer/16x1/256/1/ragged"),
    ("layer", "f32", 8, 128, "norm_rows/layer/32x1/256/1/exact"),
    ("layer", "f32", 3, 116, "norm_rows/layer/32x1/256/1/ragged"),
    ("layer", "f32", 4, 256, "norm_rows/layer/64x1/256/1/exact"),
    ("layer", "f32", 3, 244, "norm_rows/layer/64x1/256/1/ragged"),
    ("layer", "f32", 3, 500, "norm_rows_tail/layer/64x2/256/1"),
    ("layer", "f32", 3, 768, "norm_rows_tail/layer/64x3/64/1"),
    ("layer", "f32", 3, 1280, "norm_rows_tail/layer/64x5/64/1"),
    ("layer", "f32", 3, 4096, "norm_rows/layer/256x4/256/1/exact"),
    ("layer", "f32", 3, 2304, "norm_rows/layer/256x4/256/1/ragged"),
    ("layer", "f32", 3, 8192, "norm_rows/layer/256x8/256/1/exact"),
    ("layer", "f32", 3, 5120, "norm_rows/layer/256x8/256/1/ragged"),
    ("layer", "f32", 3, 16384, "norm_rows/layer/1024x4/1024/1/exact"),
    ("layer", "f32", 3, 16372, "norm_rows/layer/1024x4/1024/1/ragged"),
    ("layer", "f32", 3, 32768, "norm_rows/layer/1024x8/1024/1/exact"),
    ("layer", "f32", 3, 32756, "norm_rows/layer/1024x8/1024/1/ragged"),
    ("layer", "f32", 3, 1027, "norm_generic/layer"),
    ("rms", "f32", 3, 20, "norm_rows/rms/8x1/256/1/ragged"),
    ("rms", "f32", 3, 52, "norm_rows/rms/16x1/256/1/ragged"),
    ("rms", "f32", 3, 116, "norm_rows/rms/32x1/256/1/ragged"),
    ("rms", "f32", 3, 244, "norm_rows/rms/64x1/256/1/ragged"),
    ("rms", "f32", 3, 500, "norm_rows_tail/rms/64x2/256/1"),
    ("rms", "f32", 3, 768, "norm_rows_tail/rms/64x3/64/1"),
    ("rms", "f32", 3, 1280, "norm_rows_tail/rms/64x5/64/1"),
    ("rms", "f32", 3, 2304, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "f32", 3, 5120, "norm_rows/rms/256x8/256/1/ragged"),
    ("rms", "f32", 3, 16372, "norm_rows/rms/1024x4/1024/1/ragged"),
    ("rms", "f32", 3, 32756, "norm_rows/rms/1024x8/1024/1/ragged"),
    ("rms", "f32", 3, 1027, "norm_generic/rms"),
    ("rms", "f32", 32, 64, "norm_rows/rms/16x1/256/1/ragged"),
    ("rms", "f32", 16, 128, "norm_rows/rms/32x1/256/1/ragged"),
    ("rms", "f32", 8, 256, "norm_rows/rms/64x1/256/1/ragged"),
    ("rms", "f32", 4, 512, "norm_rows_tail/rms/64x2/256/1"),
    ("rms", "f32", 4, 768, "norm_rows_tail/rms/64x3/64/1"),
    ("rms", "f32", 4, 1280, "norm_rows_tail/rms/64x5/64/1"),
    ("rms", "f32", 4, 1536, "norm_rows_tail/rms/64x6/64/1"),
    ("rms", "f32", 4, 1792, "norm_rows_tail/rms/64x7/64/1"),
    ("rms", "f32", 4, 2048, "norm_rows_tail/rms/64x8/64/1"),
    ("rms", "f32", 4, 2304, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "f32", 4, 2560, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "f32", 4, 3072, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "f32", 4, 3584, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "f32", 4, 4096, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "f32", 4, 5120, "norm_rows/rms/256x8/256/1/ragged"),
    ("rms", "f32", 4, 6144, "norm_rows/rms/256x8/256/1/ragged"),
    ("rms", "f32", 4, 7168, "norm_rows/rms/256x8/256/1/ragged"),
    ("rms", "f32", 4, 8192, "norm_rows/rms/256x8/256/1/ragged"),
    ("layer", "f32", 32, 64, "norm_rows/layer/16x1/256/1/exact"),
    ("layer", "f32", 16, 128, "norm_rows/layer/32x1/256/1/exact"),
    ("layer", "f32", 8, 256, "norm_rows/layer/64x1/256/1/exact"),
    ("layer", "f32", 4, 512, "norm_rows_tail/layer/64x2/256/1"),
    ("layer", "f32", 4, 768, "norm_rows_tail/layer/64x3/64/1"),
    ("layer", "f32", 4, 1024, "norm_rows_tail/layer/64x4/64/1"),
    ("layer", "f32", 4, 1280, "norm_rows_tail/layer/64x5/64/1"),
    ("layer", "f32", 4, 1536, "norm_rows_tail/layer/64x6/64/1"),
    ("layer", "f32", 4, 1792, "norm_rows_tail/layer/64x7/64/1"),
    ("layer", "f32", 4, 2048, "norm_rows_tail/layer/64x8/64/1"),
    ("layer", "f32", 4, 2304, "norm_rows/layer/256x4/256/1/ragged"),
    ("layer", "f32", 4, 2560, "norm_rows/layer/256x4/256/1/ragged"),
    ("layer", "f32", 4, 3072, "norm_rows/layer/256x4/256/1/ragged"),
    ("layer", "f32", 4, 3584, "norm_rows/layer/256x4/256/1/ragged"),
    ("layer", "f32", 4, 4096, "norm_rows/layer/256x4/256/1/exact"),
    ("layer", "f32", 4, 5120, "norm_rows/layer/256x8/256/1/ragged"),
    ("layer", "f32", 4, 6144, "norm_rows/layer/256x8/256/1/ragged"),
    ("layer", "f32", 4, 7168, "norm_rows/layer/256x8/256/1/ragged"),
    ("layer", "f32", 4, 8192, "norm_rows/layer/256x8/256/1/exact"),
    ("layer", "bf16", 32, 64, "norm_rows/layer/8x1/256/1/exact"),
    ("layer", "bf16", 3, 40, "norm_rows/layer/8x1/256/1/ragged"),
    ("layer", "bf16", 16, 128, "norm_rows/layer/16x1/256/1/exact"),
    ("layer", "bf16", 3, 104, "norm_rows/layer/16x1/256/1/ragged"),
    ("layer", "bf16", 8, 256, "norm_rows/layer/32x1/256/1/exact"),
    ("layer", "bf16", 3, 232, "norm_rows/layer/32x1/256/1/ragged"),
    ("layer", "bf16", 4, 512, "norm_rows/layer/64x1/256/1/exact"),
    ("layer", "bf16", 3, 488, "norm_rows/layer/64x1/256/1/ragged"),
    ("layer", "bf16", 3, 1000, "norm_rows_tail/layer/64x2/256/1"),
    ("layer", "bf16", 3, 1536, "norm_rows_tail/layer/64x3/64/1"),
    ("layer", "bf16", 3, 2560, "norm_rows_tail/layer/64x5/64/1"),
    ("layer", "bf16", 3, 8192, "norm_rows/layer/256x4/256/1/exact"),
    ("layer", "bf16", 3, 4608, "norm_rows/layer/256x4/256/1/ragged"),
    ("layer", "bf16", 3, 16384, "norm_rows/layer/256x8/256/1/exact"),
    ("layer", "bf16", 3, 10240, "norm_rows/layer/256x8/256/1/ragged"),
    ("layer", "bf16", 3, 32768, "norm_rows/layer/1024x4/1024/1/exact"),
    ("layer", "bf16", 3, 32744, "norm_rows/layer/1024x4/1024/1/ragged"),
    ("layer", "bf16", 3, 65536, "norm_rows/layer/1024x8/1024/1/exact"),
    ("layer", "bf16", 3, 65512, "norm_rows/layer/1024x8/1024/1/ragged"),
    ("layer", "bf16", 3, 1027, "norm_generic/layer"),
    ("rms", "bf16", 3, 40, "norm_rows/rms/8x1/256/1/ragged"),
    ("rms", "bf16", 3, 104, "norm_rows/rms/16x1/256/1/ragged"),
    ("rms", "bf16", 3, 232, "norm_rows/rms/32x1/256/1/ragged"),
    ("rms", "bf16", 3, 488, "norm_rows/rms/64x1/256/1/ragged"),
    ("rms", "bf16", 3, 1000, "norm_rows_tail/rms/64x2/256/1"),
    ("rms", "bf16", 3, 1536, "norm_rows_tail/rms/64x3/64/1"),
    ("rms", "bf16", 3, 2560, "norm_rows_tail/rms/64x5/64/1"),
    ("rms", "bf16", 3, 4608, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "bf16", 3, 10240, "norm_rows/rms/256x8/256/1/ragged"),
    ("rms", "bf16", 3, 32744, "norm_rows/rms/1024x4/1024/1/ragged"),
    ("rms", "bf16", 3, 65512, "norm_rows/rms/1024x8/1024/1/ragged"),
    ("rms", "bf16", 3, 1027, "norm_generic/rms"),
    ("rms", "bf16", 32, 128, "norm_rows/rms/16x1/256/1/ragged"),
    ("rms", "bf16", 16, 256, "norm_rows/rms/32x1/256/1/ragged"),
    ("rms", "bf16", 8, 512, "norm_rows/rms/64x1/256/1/ragged"),
    ("rms", "bf16", 4, 1024, "norm_rows_tail/rms/64x2/256/1"),
    ("rms", "bf16", 4, 1536, "norm_rows_tail/rms/64x3/64/1"),
    ("rms", "bf16", 4, 2560, "norm_rows_tail/rms/64x5/64/1"),
    ("rms", "bf16", 4, 3072, "norm_rows_tail/rms/64x6/64/1"),
    ("rms", "bf16", 4, 3584, "norm_rows_tail/rms/64x7/64/1"),
    ("rms", "bf16", 4, 4096, "norm_rows_tail/rms/64x8/64/1"),
    ("rms", "bf16", 4, 4608, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "bf16", 4, 5120, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "bf16", 4, 6144, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "bf16", 4, 7168, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "bf16", 4, 8192, "norm_rows/rms/256x4/256/1/ragged"),
    ("rms", "bf16", 4, 10240, "norm_rows/rms/256x8/256/1/ragged"),
    ("rms", "bf16", 4, 12288, "norm_rows/rms/256x8/256/1/ragged"),
    ("rms", "bf16", 4, 14336, "norm_rows/rms/256x8/256/1/ragged"),
    ("rms", "bf16", 4, 16384, "norm_rows/rms/256x8/256/1/ragged"),
    ("layer", "bf16", 32, 128, "norm_rows/layer/16x1/256/1/exact"),
    ("layer", "bf16", 16, 256, "norm_rows/layer/32x1/256/1/exact"),
    ("layer", "bf16", 8, 512, "norm_rows/layer/64x1/256/1/exact"),
    ("layer", "bf16", 4, 1024, "norm_rows_tail/layer/64x2/256/1"),
    ("layer", "bf16", 4, 1536, "norm_rows_tail/layer/64x3/64/1"),
    ("layer", "bf16", 4, 2048, "norm_rows_tail/layer/64x4/64/1"),
    ("layer", "bf16", 4, 2560, "norm_rows_tail/layer/64x5/64/1"),
    ("layer", "bf16", 4, 3072, "norm_rows_tail/layer/64x6/64/1"),
    ("layer", "bf16", 4, 3584, "norm_rows_tail/layer/64x7/64/1"),
    ("layer", "bf16", 4, 4096, "norm_rows_tail/layer/64x8/64/1"),
    ("layer", "bf16", 4, 4608, "norm_rows/layer/256x4/256/1/ragged"),
    ("layer", "bf16", 4, 5120, "norm_rows/layer/256x4/256/1/ragged"),
    ("layer", "bf16", 4, 6144, "norm_rows/layer/256x4/256/1/ragged"),
    ("layer", "bf16", 4, 7168, "norm_rows/layer/256x4/256/1/ragged"),
    ("layer", "bf16", 4, 8192, "norm_rows/layer/256x4/256/1/exact"),
    ("layer", "bf16", 4, 10240, "norm_rows/layer/256x8/256/1/ragged"),
    ("layer", "bf16", 4, 12288, "norm_rows/layer/256x8/256/1/ragged"),
    ("layer", "bf16", 4, 14336, "norm_rows/layer/256x8/256/1/ragged"),
    ("layer", "bf16", 4, 16384, "norm_rows/layer/256x8/256/1/exact"),
]

# One wave per row (norm_tail.h): widths on both sides of a lane's last vector, few rows, and for two rows per wave an
# odd number of them in 20 to 64 MB.
for _k in range(2, 13):
    for _operator in ("layer", "rms"):
        _shape = f"norm_rows_tail/{_operator}/64x{_k}/" + ("256/1" if _k == 2 else "64/1")
        CASES += [(_operator, "f32", 17, 256 * (_k - 1) + 4, _shape), (_operator, "bf16", 19, 512 * _k - 8, _shape)]
        if _k > 2 and (_operator, _k) != ("rms", 4):
            CASES.append((_operator, "f32", (21 << 18) // (256 * _k - 4) | 1, 256 * _k - 4, f"norm_rows_tail/{_operator}/64x{_k}/64/2"))
CASES += [("rms", "f32", 1, 1024, "norm_rows_tail/rms/64x4/64/1"), ("layer", "bf16", 1, 1032, "norm_rows_tail/layer/64x3/64/1"),
          ("layer", "bf16", 5, 1536, "norm_rows_tail/layer/64x3/64/1"), ("rms", "bf16", 4097, 2568, "norm_rows_tail/rms/64x6/64/2"),
          ("rms", "bf16", 4001, 5640, "norm_rows_tail/rms/64x12/64/2")]
# Both sides of its rules: launches a little larger than what finds room at once (2048 blocks of four rows up to 20 MiB, 5120
# waves), rows for two rows a wave, few rows of nine narrow vectors.
CASES += [("layer", "f32", 6144, 400, "norm_rows_tail/layer/64x2/256/1"), ("layer", "f32", 6145, 400, "norm_rows/layer/64x2/256/2/ragged"),
          ("rms", "f32", 8192, 400, "norm_rows_tail/rms/64x2/256/1"), ("layer", "bf16", 8193, 800, "norm_rows/layer/64x2/256/2/ragged"),
          ("rms", "f32", 13107, 400, "norm_rows/rms/64x2/256/2/ragged"), ("rms", "bf16", 13108, 800, "norm_rows_tail/rms/64x2/256/1"),
          ("layer", "bf16", 5120, 1600, "norm_rows_tail/layer/64x4/64/1"), ("layer", "bf16", 5121, 1600, "norm_rows/layer/64x4/64/2/ragged"),
          ("layer", "bf16", 6656, 1600, "norm_rows/layer/64x4/64/2/ragged"), ("layer", "bf16", 6657, 1600, "norm_rows_tail/layer/64x4/64/1"),
          ("layer", "f32", 3999, 516, "norm_rows_tail/layer/64x3/64/1"), ("layer", "f32", 4001, 516, "norm_rows_tail/layer/64x3/64/2"),
          ("rms", "f32", 3999, 1000, "norm_rows_tail/rms/64x4/64/1"), ("rms", "f32", 4001, 1000, "norm_rows/rms/64x4/256/2/ragged"),
          ("rms", "bf16", 6999, 1032, "norm_rows_tail/rms/64x3/64/1"), ("rms", "bf16", 7001, 1032, "norm_rows_tail/rms/64x3/64/2"),
          ("rms", "bf16", 31, 4104, "norm_rows_tail/rms/64x9/64/1"), ("rms", "bf16", 33, 4104, "norm_rows/rms/256x4/256/1/ragged"),
          ("rms", "bf16", 8193, 800, "norm_rows/rms/64x2/256/2/ragged"), ("rms", "bf16", 7001, 1544, "norm_rows/rms/64x4/256/2/ragged"),
          ("layer", "bf16", 575, 4104, "norm_rows/layer/256x4/256/1/ragged"), ("layer", "bf16", 577, 4104, "norm_rows_tail/layer/64x9/64/1")]

# Few rows of up to 512 vectors a wave each, and both sides of the 10 MiB below which rows are not taken two or four to a wave.
CASES += [("rms", "f32", 2, 2048, "norm_rows_tail/rms/64x8/64/1"), ("layer", "bf16", 1, 4096, "norm_rows_tail/layer/64x8/64/1"),
          ("rms", "bf16", 2, 1536, "norm_rows_tail/rms/64x3/64/1"), ("layer", "f32", 5, 1280, "norm_rows_tail/layer/64x5/64/1"),
          ("rms", "bf16", 6, 5120, "norm_rows/rms/256x4/256/1/ragged"), ("layer", "f32", 8, 4096, "norm_rows/layer/256x4/256/1/exact"),
          ("layer", "f32", 6, 5120, "norm_rows/layer/256x8/256/1/ragged"), ("rms", "bf16", 8, 1024, "norm_rows_tail/rms/64x2/256/1"),
          ("rms", "bf16", 10232, 512, "norm_rows/rms/64x1/256/1/ragged"), ("rms", "bf16", 10240, 512, "norm_rows_exact/rms/32x2/64/4"),
          ("layer", "f32", 10232, 256, "norm_rows/layer/64x1/256/1/exact"), ("layer", "f32", 2046, 1280, "norm_rows_tail/layer/64x5/64/1"),
          ("layer", "f32", 2048, 1280, "norm_rows_exact/layer/64x5/64/2")]

# The shapes that cover the tensor exactly: 16-byte vectors to a row, shape, rows to a block; they serve from 10 MiB on.
EXACT_SHAPES = [(16, "8x2/64/4", 32), (32, "16x2/64/4", 16), (64, "32x2/64/4", 8), (128, "64x2/64/4", 4)]
EXACT_SHAPES += [(64 * _k, f"64x{_k}/64/2", 2) for _k in (3, 4, 5, 6, 7, 8, 9, 10, 12)]
EXACT_SHAPES += [(128 * _k, f"128x{_k}/128/2", 2) for _k in (7, 8)] + [(256 * _k, f"256x{_k}/256/2", 2) for _k in (5, 6, 7, 8)]
EXACT_BLOCKS = {}   # case: rows to a block
for _vectors, _shape, _block in EXACT_SHAPES:
    _rows = -((-10 << 20) // (16 * _vectors * _block)) * _block   # the fewest whole blocks of 10 MiB
    for _operator in ("layer", "rms"):
        if (_operator, _vectors) != ("rms", 256):                 # norm.hip's
            EXACT_BLOCKS.update({(_operator, _tag, _rows, _vectors * (4 if _tag == "f32" else 8), f"norm_rows_exact/{_operator}/{_shape}"): _block
                                 for _tag in ("f32", "bf16")})
CASES += list(EXACT_BLOCKS)

reached = set()


def run_case(operator, tag, weight_tag, rows, width, label, parameters, seed, distinct=None):
    """parameters: 0 none, 1 scale, 2 scale and bias (LayerNorm only).  distinct: that many rows over and over, the first of
    each held against the oracle and the others against those, bit by bit (a row's sums do not depend on its place)."""
    oid, wid = TYPES[tag][1], TYPES[weight_tag][1]
    rng = np.random.default_rng(seed)
    own = distinct or rows
    values = (rng.normal(0, 1, (own, width)) * rng.uniform(0.1, 10, (own, 1))).astype(np.float32)
    if rows > 1 and operator == "rms":
        values[1] = 2.0   # a constant row (tests/compute_provider_native/normalization_test.cc:186-199)
    xs = host_values(values, tag)
    scale = host_values(rng.normal(1, 0.1, width).astype(np.float32), weight_tag)
    bias = host_values(rng.normal(0, 0.5, width).astype(np.float32), weight_tag)
    note(f"{operator} norm {tag}/{weight_tag} [{rows}, {width}] parameters={parameters}: expecting {label}")
    operands = [to_device(xs, tag)]
    if distinct:
        operands[0] = operands[0].repeat(((rows + own - 1) // own, 1))[:rows].contiguous()
    if parameters >= 1:
        operands.append(to_device(scale, weight_tag))
    if parameters == 2:
        operands.append(to_device(bias, weight_tag))
    if operator == "rms":
        (out,) = run(hc.RmsNorm(epsilon=1e-6), *operands)
        want = orc.rms_norm(oid, xs, scale if parameters else None, 1e-6, weight_type=wid if parameters else None)
    else:
        (out,) = run(hc.LayerNorm(epsilon=1e-5), *operands)
        want = orc.layer_norm(oid, xs, scale if parameters else None, bias if parameters == 2 else None, 1e-5,
                              param_type=wid if parameters else None)
    chosen = hc.last_launch_variant()
    if label is None:
        assert not chosen.startswith("norm_rows_exact"), f"{operator} [{rows}, {width}] {tag}: launched {chosen}"
    else:
        assert chosen == label, f"{operator} [{rows}, {width}] {tag}: launched {chosen}, the table says {label}"
        reached.add(chosen)
    if distinct:
        bits = out.view(torch.int32 if tag == "f32" else torch.int16)
        assert torch.equal(bits[own:], bits[:-own]), f"{operator} [{rows}, {width}] {tag}: equal rows, other results"
    got = to_host(out[:own])
    if operator == "layer":
        layer_bar(got, want, tag, bias if parameters == 2 else None)
    elif tag == "f32":
        assert_close_f32(got, want, rel=1e-5)
    else:
        assert_narrow_ulp(got, want, tag)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}x{c[3]}")
def test_norm_case_reaches_its_launch_shape_and_matches_the_oracle(case):
    """An exact shape at the fewest rows that it serves, of which 61 are distinct, leaves a block's rows fewer to another."""
    operator, tag, rows, width, label = case
    seed = 3000 + CASES.index(case)
    distinct = 61 if case in EXACT_BLOCKS else None
    for parameters in ((0, 1) if operator == "rms" else (0, 1, 2)):
        run_case(operator, tag, tag, rows, width, label, parameters, seed + parameters, distinct)
    if tag == "bf16":   # f32 parameters under narrow storage (the cast + norm + cast of the decoder graph), and f16
        run_case(operator, "bf16", "f32", rows, width, label, 2 if operator == "layer" else 1, seed + 7, distinct)
        run_case(operator, "f16", "f16", rows, width, label, 1, seed + 8, distinct)
    if case in EXACT_BLOCKS:
        run_case(operator, tag, tag, rows - EXACT_BLOCKS[case], width, None, 1, seed, distinct)


def test_every_norm_launch_shape_in_the_library_is_reached():
    """Runs after the cases above (file order): a norm launch shape compiled into the library that no
    case reached is either dead code or an untested kernel."""
    compiled = {label for label in hc.launch_variants() if label.startswith("norm")}
    tabled = {case[4] for case in CASES}
    assert compiled == tabled, f"not in the table: {sorted(compiled - tabled)}; not in the library: {sorted(tabled - compiled)}"
    if reached:
        assert tabled <= reached, f"tabled but not reached: {sorted(tabled - reached)}"


@pytest.mark.parametrize("width", [3584, 4096, 6144, 8192])
def test_layer_norm_of_small_launches_is_no_further_from_64_bits(width):
    """f32 rows about a mean of 3, whose sums round at the size of the whole row: the shapes that serve below 10 MiB against
    those of the same rows repeated to 10 MiB, both against float64 over the same values.  800 rows leave a 2-norm within a tenth:
    a row's error is mostly its mean's, and 800 even distributions give their root mean square within 0.05 (three standard
    deviations), on either side.  (With a row's four waves added one after another 1.13 and 1.10 at 3584 and 4096.)"""
    rows = -(-(10 << 20) // (4 * width))
    rows += rows % 2
    part = (9 << 20) // (4 * width)                    # rows to a launch of less than 10 MiB
    generator = torch.Generator(device="cuda:0").manual_seed(5500 + width)
    x = torch.randn((800, width), device="cuda:0", generator=generator) + 3.0
    note(f"layer norm f32 [800, {width}] about 3: {part} rows at a time, and among {rows}")
    wide = x.double()
    wide = wide - wide.mean(1, keepdim=True)
    want = wide / (wide.pow(2).mean(1, keepdim=True) + 1e-5).sqrt()
    off = []
    for step, family in ((part, "norm_rows/layer/256"), (rows, "norm_rows_exact/layer/")):
        got = []
        for first in range(0, 800, step):
            piece = x[first:first + step]
            held = len(piece)
            if step == rows:
                piece = piece.repeat((rows + held - 1) // held, 1)[:rows].contiguous()
            (out,) = run(hc.LayerNorm(epsilon=1e-5), piece)
            assert hc.last_launch_variant().startswith(family), hc.last_launch_variant()
            got.append(out[:held])
        off.append((torch.cat(got).double() - want).norm().item())
    assert off[0] <= 1.1 * off[1], f"{off[0] / off[1]:.3f}"
