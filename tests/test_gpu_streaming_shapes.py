"""The launch shapes of the streaming kernels that depend on a launch's traffic: sizes on both sides of each line, odd
ones among them.  Sums, conversions and moves of 32-bit words are exact, so numpy is the reference."""
from __future__ import annotations

import numpy as np
import pytest

from hyle_amd import compute as hc

from gpu_support import assert_bits_equal, last_launch_form, note, run, to_device, to_host

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.mark.parametrize("elements,shape", [
    (1, "1x64/batched"), (255, "1x64/batched"), (4097, "1x64/batched"), (42 * MIB // 12, "1x64/batched"),
    (42 * MIB // 12 + 3, "4x512/serial"), (48 * MIB // 12, "4x512/serial"), (48 * MIB // 12 + 5, "1x64/batched")])
def test_add_of_whole_operands(elements, shape):
    rng = np.random.default_rng(elements)
    a, b = rng.normal(0, 1, (2, elements)).astype(np.float32)
    note(f"binary add f32 [{elements}]")
    (out,) = run(hc.Binary(hc.BinaryKind.kAdd), to_device(a, "f32"), to_device(b, "f32"))
    assert hc.last_launch_variant() == "ew_full/" + shape
    assert_bits_equal(to_host(out), a + b)


@pytest.mark.parametrize("rows,shape", [(2, "1x256"), (3071, "1x256"), (3072, "4x1024"), (10240, "4x1024"), (10241, "1x256")])
def test_add_of_a_row(rows, shape):
    rng = np.random.default_rng(rows)
    a, b = rng.normal(0, 1, (rows, 1024)).astype(np.float32), rng.normal(0, 1, 1024).astype(np.float32)
    note(f"binary add f32 [{rows}, 1024] + [1024]")
    (out,) = run(hc.Binary(hc.BinaryKind.kAdd), to_device(a, "f32"), to_device(b, "f32"))
    assert hc.last_launch_variant() == "ew_flat/" + shape
    assert_bits_equal(to_host(out), a + b)


@pytest.mark.parametrize("elements,shape", [
    (7, "1x256/batched"), (24 * MIB // 8, "1x256/batched"), (24 * MIB // 8 + 1, "4x512/serial"), (48 * MIB // 8, "4x512/serial"),
    (48 * MIB // 8 + 3, "8x512/serial"), (110 * MIB // 8, "8x512/serial"), (110 * MIB // 8 + 2, "1x64/batched")])
def test_dense_copy(elements, shape):
    words = np.random.default_rng(elements).integers(0, 1 << 32, elements, dtype=np.uint32)
    note(f"copy of {elements} words")
    (out,) = run(hc.Copy(), to_device(words.view(np.float32), "f32"))
    assert hc.last_launch_variant() == "cast_flat/" + shape
    assert np.array_equal(to_host(out).view(np.uint32), words)


# below 16 MiB of output one unit per thread, four up to 64 MiB, two in smaller blocks above; runs that end inside a block
@pytest.mark.parametrize("outer,first,second,inner", [(3, 5, 1, 4), (7, 301, 999, 64), (5, 8192, 700, 80), (16, 3072, 1000, 128), (9, 8000, 300, 256)])
def test_concat_runs(outer, first, second, inner):
    rng = np.random.default_rng(inner)
    a, b = (rng.normal(0, 1, (outer, n, inner)).astype(np.float32) for n in (first, second))
    note(f"concat [{outer}, {first} + {second}, {inner}]")
    (out,) = run(hc.Concat(1), to_device(a, "f32"), to_device(b, "f32"))
    assert hc.last_launch_variant() == "concat_runs/16-bytes"
    assert_bits_equal(to_host(out), np.concatenate([a, b], axis=1))


# outputs on both sides of 15 and 64 MiB, runs on both sides of 16 KiB, many short ones; units of every width have four to a
# thread at any size
@pytest.mark.parametrize("outer,first,second,inner,form", [
    (3, 5, 1, 4, "16-bytes#1x256"), (4, 7679, 7680, 64, "16-bytes#1x256"), (4, 7680, 7680, 64, "16-bytes#4x256"), (1, 1, 1 << 16, 64, "16-bytes#4x256"),
    (4, 32767, 32768, 64, "16-bytes#4x256"), (4, 32768, 32768, 64, "16-bytes#2x128"), (9, 8000, 1333, 256, "16-bytes#2x128"),
    (70, 16, 1000, 256, "16-bytes#2x128"), (70, 15, 1000, 256, "16-bytes#4x256"), (1023, 3, 2, 52, "16-bytes#1x256"), (1024, 3, 2, 52, "16-bytes#4x256"),
    (5, 2, 7, 1001, "4-bytes#4x256"), (3, 70000, 30001, 67, "4-bytes#4x256")])
def test_concat_runs_in_every_form(outer, first, second, inner, form):
    rng = np.random.default_rng(first)
    a, b = (rng.integers(0, 1 << 32, (outer, n, inner), dtype=np.uint32).view(np.float32) for n in (first, second))
    note(f"concat [{outer}, {first} + {second}, {inner}]: {form}")
    (out,) = run(hc.Concat(1), to_device(a, "f32"), to_device(b, "f32"))
    assert last_launch_form() == "concat_runs/" + form
    assert np.array_equal(to_host(out).view(np.uint32), np.concatenate([a, b], axis=1).view(np.uint32))
