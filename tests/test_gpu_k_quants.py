"""GGUF Q4_K / Q6_K rows -> bf16 + row sums of squares (through the C ABI) against the oracle:
bit-exact bf16 values, sums of squares within 1e-5 relative.  The blocks come from the field-wise
builders of tests/k_quant_support.py and from raw random bytes (any byte pattern is a valid block
as long as its f16 scales are finite)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from hyle_amd import compute as hc
from oracle import lib as orc

from gpu_support import DEVICE, context, note, run
from k_quant_support import random_rows

pytestmark = pytest.mark.gpu

KINDS = {"q4_k": (orc.Q4_K, hc.GgufQuantizedType.kQ4K, 144), "q6_k": (orc.Q6_K, hc.GgufQuantizedType.kQ6K, 210)}


def dequant_on_device(tag, raw, rows, k, row_stride=None, offset=0):
    _, gguf, _ = KINDS[tag]
    storage = torch.from_numpy(np.ascontiguousarray(raw).reshape(-1)).to(DEVICE)
    desc = hc.TensorDesc.gguf_weight(gguf, hc.DataType.kBFloat16, k, rows, row_stride)
    out, sumsq = run(hc.GgufDequantSumSquares(), storage[offset:], descs=[desc])
    return out.contiguous().view(torch.int16).cpu().numpy().view(np.uint16), sumsq.cpu().numpy()


def sumsq_bar(got, wide):
    """Row sums of squares against the float64 sum of the oracle's exact f32 values: 1e-5 relative.
    (The oracle's own sequential f32 sum is a looser witness: 2048 heavy-tailed terms.)"""
    exact = np.sum(wide.astype(np.float64) ** 2, axis=1)
    assert np.all(np.abs(got.astype(np.float64) - exact) <= 1e-5 * exact)


def finite_scales(tag, raw, block_bytes):
    """Random bytes with the f16 fields forced finite."""
    blocks = raw.reshape(-1, block_bytes)
    for at in ((1, 3) if tag == "q4_k" else (209,)):
        blocks[:, at] &= 0x3B            # exponent below all-ones, small magnitude
    return raw


@pytest.mark.parametrize("tag", ["q4_k", "q6_k"])
def test_k_quant_built_blocks_and_random_bytes(tag):
    kind, _, block_bytes = KINDS[tag]
    rng = np.random.default_rng(1500)
    for rows, k in ((1, 256), (3, 768), (5, 2048), (2, 2304), (4, 4096)):
        raw, values = random_rows(tag, rng, rows, k)
        note(f"{tag} built blocks [{rows}, {k}]")
        got, sumsq = dequant_on_device(tag, raw, rows, k)
        wide, want, want_sumsq = orc.k_quant_dequant(kind, raw, rows, k)
        assert np.array_equal(wide, values)                      # the oracle against the builders
        assert np.array_equal(got, want)
        sumsq_bar(sumsq, wide)
        assert np.allclose(want_sumsq, np.sum(wide.astype(np.float64) ** 2, axis=1), rtol=2e-4)
        note(f"{tag} random bytes [{rows}, {k}]")
        raw = finite_scales(tag, rng.integers(0, 256, (rows, k // 256 * block_bytes), dtype=np.uint8), block_bytes)
        got, sumsq = dequant_on_device(tag, raw, rows, k)
        wide, want, want_sumsq = orc.k_quant_dequant(kind, raw, rows, k)
        assert np.array_equal(got, want)
        sumsq_bar(sumsq, wide)


@pytest.mark.parametrize("tag", ["q4_k", "q6_k"])
def test_k_quant_padded_rows_and_odd_addresses(tag):
    kind, _, block_bytes = KINDS[tag]
    rng = np.random.default_rng(1501)
    rows, k = 6, 1024
    row_bytes = k // 256 * block_bytes
    raw = finite_scales(tag, rng.integers(0, 256, (rows, row_bytes), dtype=np.uint8), block_bytes)
    wide, want, want_sumsq = orc.k_quant_dequant(kind, raw, rows, k)
    for pad, offset in ((2, 0), (7, 0), (0, 1), (5, 3), (16, 2)):
        padded = np.zeros(offset + rows * (row_bytes + pad) + 8, np.uint8)
        for r in range(rows):
            start = offset + r * (row_bytes + pad)
            padded[start:start + row_bytes] = raw[r]
        note(f"{tag} rows {row_bytes + pad} bytes apart, tensor at byte {offset}")
        got, sumsq = dequant_on_device(tag, padded, rows, k, row_stride=row_bytes + pad, offset=offset)
        assert np.array_equal(got, want)
        sumsq_bar(sumsq, wide)


@pytest.mark.parametrize("tag", ["q4_k", "q6_k"])
def test_k_quant_whole_vector_rows(tag):
    """K a multiple of 2048 with base and row stride multiples of 16 takes the wave-per-row kernel
    (several spans per row, padded strides, a row count that leaves waves of the last block idle);
    the same rows 2 bytes off take the general one."""
    kind, _, block_bytes = KINDS[tag]
    rng = np.random.default_rng(1503)
    for rows, k in ((7, 2048), (13, 6144), (257, 4096)):
        row_bytes = k // 256 * block_bytes
        raw = finite_scales(tag, rng.integers(0, 256, (rows, row_bytes), dtype=np.uint8), block_bytes)
        wide, want, _ = orc.k_quant_dequant(kind, raw, rows, k)
        for pad, offset in ((0, 0), (16, 0), (48, 32), (16, 2)):
            padded = np.zeros(offset + rows * (row_bytes + pad) + 8, np.uint8)
            for r in range(rows):
                start = offset + r * (row_bytes + pad)
                padded[start:start + row_bytes] = raw[r]
            note(f"{tag} [{rows}, {k}] rows {row_bytes + pad} bytes apart, tensor at byte {offset}")
            got, sumsq = dequant_on_device(tag, padded, rows, k, row_stride=row_bytes + pad, offset=offset)
            assert np.array_equal(got, want)
            sumsq_bar(sumsq, wide)


def test_k_quant_schema_and_benchmark_shape():
    DT = hc.DataType
    desc = hc.TensorDesc.gguf_weight(hc.GgufQuantizedType.kQ4K, DT.kBFloat16, 2048, 6144)
    values, sumsq = hc.infer_output_descriptions(hc.GgufDequantSumSquares(), [desc])
    assert values == hc.TensorDesc.dense(DT.kBFloat16, [6144, 2048]) and sumsq == hc.TensorDesc.dense(DT.kFloat32, [6144])
    assert hc.prepare(context(), hc.GgufDequantSumSquares(), desc).route_name() == "k-quant-dequant-rows"
    with pytest.raises(hc.StatusError):
        hc.TensorDesc.gguf_weight(hc.GgufQuantizedType.kQ6K, DT.kBFloat16, 2000, 8)
    rng = np.random.default_rng(1502)
    for tag in ("q4_k", "q6_k"):
        kind, _, block_bytes = KINDS[tag]
        raw = finite_scales(tag, rng.integers(0, 256, (6144, 8 * block_bytes), dtype=np.uint8), block_bytes)
        note(f"{tag} [6144, 2048]")
        got, sumsq = dequant_on_device(tag, raw, 6144, 2048)
        wide, want, want_sumsq = orc.k_quant_dequant(kind, raw, 6144, 2048)
        assert np.array_equal(got, want)
        sumsq_bar(sumsq, wide)


# rows, k: pieces of 2048 values that are not whole, a row to a wave and (rows of more than one piece, at most eight to a compute unit,
# of Q4_K up to seven and a half) to a block
@pytest.mark.parametrize("tag", ["q4_k", "q6_k"])
def test_k_quant_rows_of_pieces(tag):
    kind, _, block_bytes = KINDS[tag]
    rng = np.random.default_rng(1504)
    for rows, k in ((5, 256), (9, 1792), (2, 2304), (2048, 2304), (2049, 2304), (3, 4096), (7, 8448), (2051, 3840), (2050, 4096),
                    (1792, 4096), (1793, 2304), (1920, 4352), (1921, 4352), (1664, 8448), (1665, 8448)):
        row_bytes = k // 256 * block_bytes
        raw = finite_scales(tag, rng.integers(0, 256, (min(rows, 40), row_bytes), dtype=np.uint8), block_bytes)
        raw = np.resize(raw, (rows, row_bytes))
        wide, want, _ = orc.k_quant_dequant(kind, raw, rows, k)
        for pad, offset in ((0, 0), (16, 32), (16, 6), (-row_bytes % 16 + 14, 14)):
            padded = np.zeros(offset + rows * (row_bytes + pad) + 8, np.uint8)
            padded[offset:offset + rows * (row_bytes + pad)].reshape(rows, -1)[:, :row_bytes] = raw
            served = (offset | (row_bytes + pad)) % (16 if tag == "q4_k" else 2) == 0
            note(f"{tag} [{rows}, {k}] rows {row_bytes + pad} bytes apart, tensor at byte {offset}")
            got, sumsq = dequant_on_device(tag, padded, rows, k, row_stride=row_bytes + pad, offset=offset)
            halves = 16 if tag == "q6_k" else (14 if k <= 4096 else (15 if k <= 8192 else 13))
            together = torch.cuda.get_device_properties(0).multi_processor_count * halves // 2
            form = "/shared" if k > 2048 and rows <= together else ("/pieces" if k % 2048 else "")
            label = f"k_quant_lines/{tag}{form}" if served else f"k_quant_rows/{tag}"
            assert hc.last_launch_variant() == label
            assert np.array_equal(got, want)
            sumsq_bar(sumsq, wide)


@pytest.mark.parametrize("tag,rows,k", [("q4_k", 2100, 14080), ("q4_k", 2100, 17408), ("q4_k", 300, 17408), ("q4_k", 2100, 7168), ("q6_k", 2100, 17408),
                                        ("q6_k", 300, 14080), ("q6_k", 2100, 8192), ("q8_0", 300, 17408), ("q8_0", 6144, 2304), ("q8_0", 300, 8192)])
def test_row_sums_of_squares_round_seldom(tag, rows, k):
    """Against the float64 sums of the same f32 values, 2-norm over 300 distinct rows.  The last rounding moves a sum by
    2^-24 / sqrt(3) of it in root mean square, at the foot of a binade.  Each of 64 lanes adds K / 512 sums of eight squares, a
    rounding of the part there is so far each time (a third of so many whole ones in the mean square) and three whole ones at
    most within the eights, independent of the other lanes'; the first three steps over the lanes are in f32, at 1/32, 1/16
    and 1/8 of a sum.  300 rows give the mean square of an even distribution within
    0.155 of it, three standard deviations.  (One chain of squares a lane: 5.2e-8 to 7.0e-8 at these widths of Q4_K.)"""
    rng = np.random.default_rng(1506)
    distinct = 300
    if tag == "q8_0":
        blocks = rng.integers(0, 256, (distinct, k // 32, 34), dtype=np.uint8)
        blocks[:, :, 1] = blocks[:, :, 1] & 0x07 | 0x10
        raw = blocks.reshape(distinct, -1)
        wide = (blocks[:, :, 2:].view(np.int8).astype(np.float32) * blocks[:, :, :2].copy().view(np.float16).astype(np.float32)).reshape(distinct, k)
    else:
        kind, _, block_bytes = KINDS[tag]
        raw = finite_scales(tag, rng.integers(0, 256, (distinct, k // 256 * block_bytes), dtype=np.uint8), block_bytes)
        wide = orc.k_quant_dequant(kind, raw, distinct, k)[0]
    gguf = {"q8_0": hc.GgufQuantizedType.kQ8_0, "q4_k": hc.GgufQuantizedType.kQ4K, "q6_k": hc.GgufQuantizedType.kQ6K}[tag]
    desc = hc.TensorDesc.gguf_weight(gguf, hc.DataType.kBFloat16, k, rows)
    note(f"{tag} [{rows}, {k}]: row sums of squares against float64")
    _, sumsq = run(hc.GgufDequantSumSquares(), torch.from_numpy(np.resize(raw, (rows, raw.shape[1]))).to(DEVICE), descs=[desc])
    got = sumsq.cpu().numpy()
    assert np.array_equal(got, np.resize(got[:distinct], rows))
    want = (np.asarray(wide, np.float64).reshape(distinct, k) ** 2).sum(1)
    off = np.linalg.norm((got[:distinct] - want) / want) / np.sqrt(distinct)
    assert off <= np.sqrt(1.155 * (1 / 3 + (k / 512 / 3 + 3) / (3 * 64) + 7 / 32 / 3)) * 2.0 ** -24, f"{off:.3e}"


def test_q8_0_rows_of_pieces():
    """The larger ones on both sides of the launches that are resident at once on 256 compute units, where blocks stage whole rows."""
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    rng = np.random.default_rng(1505)
    for rows, k, pad, label in ((5, 256, 0, "lines/pieces"), (9, 1792, 16, "lines/pieces"), (6, 2304, 0, "lines/pieces"), (1030, 3840, 32, "lines/pieces"),
                                (5, 16640, 0, "lines/pieces"), (7, 10240, 16, "lines"), (4096, 2304, 0, "lines/pieces"), (4097, 2304, 16, "rows"),
                                (8192, 4608, 0, "rows"), (8193, 2560, 0, "lines/pieces"), (7168, 4864, 0, "rows"), (7169, 4864, 0, "lines/pieces"),
                                (3580, 7936, 0, "lines/pieces"), (3581, 7936, 32, "rows"), (4096, 9472, 0, "rows"), (4099, 8192, 0, "lines"), (5000, 9984, 0, "lines/pieces"),
                                (4, 2304, 2, "rows_bytes"), (4, 2272, 0, "rows_bytes")):
        blocks = rng.integers(0, 256, (rows, k // 32, 34), dtype=np.uint8)
        blocks[:, :, 1] &= 0x3B
        raw = blocks.reshape(rows, -1)
        padded = np.zeros((rows, raw.shape[1] + pad), np.uint8)
        padded[:, :raw.shape[1]] = raw
        desc = hc.TensorDesc.gguf_weight(hc.GgufQuantizedType.kQ8_0, hc.DataType.kBFloat16, k, rows, raw.shape[1] + pad)
        note(f"q8_0 [{rows}, {k}] rows {raw.shape[1] + pad} bytes apart")
        out, sumsq = run(hc.GgufDequantSumSquares(), torch.from_numpy(padded).to(DEVICE), descs=[desc])
        assert hc.last_launch_variant() == f"q8_0_{label}"
        values = blocks[:, :, 2:].view(np.int8).astype(np.float32) * blocks[:, :, :2].copy().view(np.float16).astype(np.float32)
        assert np.array_equal(out.contiguous().view(torch.int16).cpu().numpy().view(np.uint16), orc.from_f32(orc.BF16, values.reshape(rows, k)))
        sumsq_bar(sumsq.cpu().numpy(), values.reshape(rows, k))
