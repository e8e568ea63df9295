"""Softmax / LogSoftmax over rows that are no whole number of 16-byte vectors or start off a 16-byte
boundary: the launch shapes of softmax_unaligned.hip at both ends of the widths each one takes,
against the oracle under the bars of test_gpu_softmax_variants.py (f32 1e-5 relative, narrow types one
unit in the last place, LogSoftmax f32 4e-6 relative + 2e-7)."""
from __future__ import annotations

import pytest
import torch

from hyle_amd import compute as hc

from gpu_support import DEVICE, TYPES, last_launch_form, note, run
from test_gpu_softmax_variants import MASKS, compare_on_device, make_inputs, oracle_softmax

pytestmark = pytest.mark.gpu

# (fewest, most vectors per row, launch shape)
SHAPES = [(1, 8, "8x1/256"), (9, 16, "16x1/256"), (17, 32, "16x2/256"), (33, 64, "32x2/256"), (65, 96, "32x3/256"),
          (97, 128, "64x2/256"), (129, 192, "64x3/256"), (193, 256, "64x4/256"), (257, 384, "128x3/256"), (385, 512, "128x4/256"),
          (513, 768, "256x3/256"), (769, 1024, "256x4/256"), (1025, 1536, "512x3/512"), (1537, 2048, "512x4/512"),
          (2049, 8192, "1024x8/1024")]


def offset_by_one(t):
    """The same values one element behind a 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    flat[1:] = t.reshape(-1)
    return flat[1:].view(t.shape)


def check(tag, q, width, mask_word, shape, log_form, moved, in_place, heads=2, mask_moved=False):
    scale = 0.125 if mask_word != "unmasked" else 1.0
    note(f"softmax {tag} log={log_form} [{heads}, {q}, {width}] {mask_word} moved={moved} {mask_moved} in_place={in_place}: expecting {shape}")
    x, x_host, mask, mask_host = make_inputs(tag, heads, q, width, mask_word, seed=width + q)
    if moved:   # x, or a mask under rows that are no whole number of vectors anyway
        x = offset_by_one(x)
    if mask is not None and (moved or mask_moved):
        mask = offset_by_one(mask)
    want = oracle_softmax(tag, x_host, mask_word, mask_host, scale, log_form)
    kind = hc.SoftmaxKind.kLogSoftmax if log_form else hc.SoftmaxKind.kSoftmax
    (out,) = run(hc.Softmax(scale=scale, kind=kind, mask=MASKS[mask_word]), *([x] if mask is None else [x, mask]),
                 outputs=[x] if in_place else None)
    assert hc.last_launch_variant() == f"softmax_unaligned/{shape}/{mask_word}"
    count, text = compare_on_device(tag, out, want, log_form)
    assert count == 0, f"{count} elements outside the bar, {text}"


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: s[2].replace("/", "-"))
@pytest.mark.parametrize("tag", ["f32", "bf16", "f16"])
def test_rows_of_any_width_at_both_ends_of_a_launch_shape(shape, tag):
    fewest, most, label = shape
    vec = 16 // TYPES[tag][2].itemsize
    for width, moved in ((max(vec, (fewest - 1) * vec + 1), fewest == 1), (most * vec - 1, False), (most * vec, True)):
        q = max(5, 400 // width + 1)
        for mask_word in ("unmasked", "boolean", "additive"):
            check(tag, q, width, mask_word, label, False, moved, in_place=mask_word == "boolean")
            check(tag, q, width, mask_word, label, True, moved, in_place=False, mask_moved=True)
    # rows of whole vectors under a mask that starts one element behind a boundary
    for mask_word in ("boolean", "additive"):
        check(tag, max(5, 400 // (most * vec) + 1), most * vec, mask_word, label, False, False, in_place=False, mask_moved=True)


@pytest.mark.parametrize("tag", ["f32", "bf16", "f16"])
def test_a_few_short_rows(tag):
    """One head, one to six rows, from a single vector and one element on: no size is too small for these launch shapes."""
    vec = 16 // TYPES[tag][2].itemsize
    for q, width in ((1, vec + 1), (2, vec + 1), (1, 129), (6, 129), (1, 777), (4, 197)):
        shape = next(label for fewest, most, label in SHAPES if fewest <= (width + vec - 1) // vec <= most)
        for mask_word in ("unmasked", "boolean", "additive"):
            check(tag, q, width, mask_word, shape, False, width * q % vec == 0, in_place=False, heads=1)


@pytest.mark.parametrize("lowest", [-20.0, -85.0])
@pytest.mark.parametrize("tag", ["bf16", "f16"])
def test_narrow_rows_are_no_further_from_64_bits_than_the_strided_kernel(tag, lowest):
    """The exponentials behind a narrow result are 32-bit ones with errors below 2e-6, so few results are on the wrong side of
    a rounding; counted against float64 there must be no more of them than softmax_general gives for the same rows seen
    through a stride.  Where both exponentials are as good as each other their last bits still differ: two units of 2^-24 move
    a share of 2 * 2^-24 / 2^-8 of bf16 results across a rounding, for the better or the worse alike, so the counts may differ
    by three standard deviations of that (17; a single multiply-add into exp2 has 58 too many at bf16 down to e^-85, 20 too
    many at f16 down to e^-20)."""
    rows, width, scale = 1024, 1013, 0.7
    generator = torch.Generator(device=DEVICE).manual_seed(1840)
    x = torch.empty((rows, width), device=DEVICE).uniform_(lowest / scale, 0.0, generator=generator).to(TYPES[tag][2])
    spread = torch.zeros((rows, width, 2), dtype=x.dtype, device=DEVICE)
    spread[..., 0] = x
    exact = torch.softmax((x.float() * scale).double(), -1).to(x.dtype)   # one rounding
    note(f"softmax {tag} [{rows}, {width}] down to {lowest}: dense and strided rows against float64")
    wrong = []
    for rows_seen, label in ((x, "softmax_unaligned/"), (spread[..., 0], "softmax_general")):
        (out,) = run(hc.Softmax(scale=scale), rows_seen)
        assert hc.last_launch_variant().startswith(label)
        wrong.append(int((out.view(torch.int16) != exact.view(torch.int16)).sum()))
    assert wrong[0] <= wrong[1] + 3.0 * (rows * width * 2.0 ** -15) ** 0.5, wrong


@pytest.mark.parametrize("tag,heads,q,width,mask_word,shape", [
    ("bf16", 7, 3487, 2049, "additive", "128x3/256"), ("f16", 4, 4071, 3071, "boolean", "128x3/256"), ("f32", 5, 4864, 1031, "boolean", "128x3/256"),
    ("bf16", 8, 2036, 3073, "boolean", "128x4/256"), ("f16", 4, 3058, 4089, "additive", "128x4/256"), ("f32", 3, 4200, 2047, "additive", "128x4/256"),
    ("f16", 3, 4070, 4097, "additive", "256x3/256"), ("bf16", 5, 2001, 5001, "boolean", "256x3/256"), ("f32", 4, 2048, 3067, "additive", "256x3/256"),
    ("f16", 3, 2720, 6145, "boolean", "256x4/256"), ("bf16", 7, 900, 8191, "additive", "256x4/256"), ("f32", 3, 2200, 4091, "boolean", "256x4/256")])
def test_heads_that_share_a_mask_row(tag, heads, q, width, mask_word, shape):
    """Three heads to a block's mask row, one, two or three in the last, at both ends of each width: odd and even numbers of rows,
    in place, and LogSoftmax; a tensor below the least size, and two heads, go the other way."""
    log_form = heads % 2 == 0
    check(tag, q, width, mask_word, shape, log_form, False, in_place=not log_form, heads=heads)
    assert last_launch_form() == f"softmax_unaligned/{shape}/{mask_word}#shared"
    if (heads, width) == (4, 4089):
        for other_heads, rows in ((4, q - 2), (2, 2 * q)):
            check(tag, rows, width, mask_word, shape, False, False, in_place=False, heads=other_heads)
            assert not last_launch_form().endswith("#shared")


@pytest.mark.parametrize("tag,mask_word,q,width,shape", [("bf16", "additive", 2036, 3073, "128x4/256"), ("f32", "boolean", 2048, 3067, "256x3/256")])
@pytest.mark.parametrize("layout", ["for all", "a batch of one", "off a boundary", "a batch"])
def test_masks_shared_by_leading_axes(tag, mask_word, q, width, shape, layout):
    """[batch, heads, q, k]: a mask [q, k] for both leading axes, one whose batch axis of extent 1 has a stride of its own, one
    that starts one element behind a boundary; a mask for each batch is shared by its heads alone and no block takes three."""
    batches, heads = (1, 8) if layout == "a batch of one" else (2, 4)
    note(f"softmax {tag} [{batches}, {heads}, {q}, {width}] {mask_word}, the mask {layout}")
    x, x_host, mask, mask_host = make_inputs(tag, 8, q, width, mask_word, seed=width)
    want = oracle_softmax(tag, x_host, mask_word, mask_host, 0.125, False)
    if layout == "a batch of one":
        padded = torch.zeros((1, 1, q + 1, width), dtype=mask.dtype, device=DEVICE)
        padded[0, 0, :q] = mask
        mask = padded[:, :, :q]              # the axes of extent 1 keep the strides of q + 1 rows
        assert mask.stride(0) != q * width
    elif layout == "off a boundary":
        mask = offset_by_one(mask)
    elif layout == "a batch":
        other, other_host = make_inputs(tag, 1, q, width, mask_word, seed=width + 1)[2:]
        mask = torch.stack([mask, other])[:, None]
        want[4:] = oracle_softmax(tag, x_host[4:], mask_word, other_host, 0.125, False)
    (out,) = run(hc.Softmax(scale=0.125, mask=MASKS[mask_word]), x.view(batches, heads, q, width), mask)
    assert last_launch_form() == f"softmax_unaligned/{shape}/{mask_word}" + ("" if layout == "a batch" else "#shared")
    count, text = compare_on_device(tag, out.view(8, q, width), want, False)
    assert count == 0, f"{count} elements outside the bar, {text}"
