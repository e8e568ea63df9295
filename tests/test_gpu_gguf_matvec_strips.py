"""The GGUF products with 8-bit activation blocks against many weight rows (gguf_matvec_strips.hip):
every format, one and two sets of activation rows, both block sizes, one and two blocks per compute
unit, one to sixteen waves to a tile, rows that are no whole number of 16-byte vectors or start off a
boundary.  Bar and oracle as in test_gpu_gguf_matvec_q8.py."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from hyle_amd import compute as hc
from oracle import lib as orc

from gpu_support import DEVICE, context, note, run
from k_quant_support import pack_q6_k
from test_gpu_gguf_matvec_q8 import KINDS, Q8, check, raw_bytes_for, weights_for

pytestmark = pytest.mark.gpu

# rows, k, activation rows, bytes the weight starts off a boundary, bytes between rows, activation elements off
CASES = (
    (4096, 1280, 5, 0, 0, 0),     # five runs, split over fewer waves than a block has
    (4099, 5120, 7, 0, 0, 0),     # a last block with fewer rows, a tile with rows that repeat
    (12289, 1536, 2, 0, 0, 0),    # two blocks per compute unit
    (66000, 256, 2, 0, 0, 0),     # one run: a wave to a tile, no shares
    (5003, 1792, 4, 2, 6, 1),     # rows at every even offset, activations at an odd element
    (4097, 2048, 8, 14, 10, 3),
    (521, 12544, 8, 0, 2, 0),     # eight waves to a block
    (530, 25600, 3, 6, 0, 1),     # wide rows
)


@pytest.mark.parametrize("x_tag", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("tag", list(KINDS))
def test_strips_edges(tag, x_tag):
    rng = np.random.default_rng(1820)
    for rows, k, m, byte_offset, pad, x_offset in CASES:
        if tag == "q4_k" and not pad and not byte_offset and (k < 4096 or rows < 4096):
            byte_offset = 2   # a boundary would take the tile kernel
        raw = raw_bytes_for(tag, rng, rows, k) if x_tag != "f16" else weights_for(tag, rng, rows, k)
        padded = np.zeros((rows, raw.shape[1] + pad), np.uint8)
        padded[:, :raw.shape[1]] = raw
        x = rng.normal(0, 1.5, (m, k)).astype(np.float32)
        x[m - 1, :256] = 0.0                                                        # an activation block of zeros
        x[0, k - 256:] = np.where(np.arange(256) % 2 == 0, -1.25, 1.25)             # equal magnitudes: the first sign decides
        note(f"q8 matvec strips {tag} x {x_tag} rows {rows} k {k} m {m} off {byte_offset} pad {pad} x off {x_offset}")
        check(tag, x_tag, padded, rows, k, x, row_stride=raw.shape[1] + pad, byte_offset=byte_offset, x_offset=x_offset,
              kernel=f"gguf_matvec_q8_strips/{tag}/{4 if m <= 4 else 8}-tokens")


# rows, k, activation rows, the form: Q8_0 rows of whole vectors, whose bytes the matrix unit takes as they lie
IN_PLACE = (
    (513, 256, 2, "4-tokens/16-waves/in-place/parked"),  # one run, three weight rows to a block
    (4099, 1280, 5, "8-tokens/16-waves/shared/in-place/parked"),
    (2050, 5120, 4, "4-tokens/16-waves/shared/in-place/parked"),
    (4096, 256, 8, "8-tokens/16-waves/in-place/parked"),
    (66000, 256, 3, "4-tokens/2x8-waves/in-place/parked"),
    (66000, 256, 8, "8-tokens/2x8-waves/in-place/parked"),
    (12289, 1792, 2, "4-tokens/2x8-waves/shared/in-place/parked"),
    (9001, 1280, 7, "8-tokens/2x8-waves/shared/in-place/parked"),
    (70000, 4352, 4, "4-tokens/2x8-waves/shared/in-place/parked"),  # more tiles than waves
    (1031, 4096, 8, "8-tokens/16-waves/shared/in-place/parked"),
    (530, 25600, 3, "4-tokens/16-waves/in-place"),  # no room for slots: straight into the lanes
    (515, 28672, 3, "4-tokens/16-waves/in-place"),
    (519, 17408, 5, "8-tokens/16-waves/in-place"),
)


@pytest.mark.parametrize("x_tag", ["f32", "bf16", "f16"])
def test_strips_q8_0_in_place(x_tag):
    rng = np.random.default_rng(1823)
    for rows, k, m, form in IN_PLACE:
        raw = raw_bytes_for("q8_0", rng, rows, k) if x_tag != "f16" else weights_for("q8_0", rng, rows, k)
        padded = np.zeros((rows, raw.shape[1] + 16), np.uint8)                       # whole vectors between rows too
        padded[:, :raw.shape[1]] = raw
        x = rng.normal(0, 1.5, (m, k)).astype(np.float32)
        x[m - 1, :32], x[0, k - 32:] = 0.0, -3.0                                    # a block of zeros, one of equal values
        note(f"q8 matvec strips in place x {x_tag} rows {rows} k {k} m {m}")
        check("q8_0", x_tag, padded, rows, k, x, row_stride=raw.shape[1] + 16, kernel=f"gguf_matvec_q8_strips/q8_0/{form}")


def test_strips_decoded_q8_0_off_a_boundary_in_every_form():
    rng = np.random.default_rng(1824)
    for rows, k, m in ((66000, 256, 2), (66000, 256, 5), (12289, 1536, 2), (9001, 1280, 7), (70000, 4352, 4), (70000, 4352, 5), (4096, 1280, 5), (600, 1536, 3)):
        raw = raw_bytes_for("q8_0", rng, rows, k)
        note(f"q8 matvec strips q8_0 rows {rows} k {k} m {m}, two bytes off")
        check("q8_0", "bf16", raw, rows, k, rng.normal(0, 1, (m, k)).astype(np.float32), byte_offset=2, kernel="gguf_matvec_q8_strips/q8_0/")


@pytest.mark.parametrize("tag,k,rows,m,kernel", [
    ("q6_k", 2304, 24000, 1, "strips/q6_k/4"), ("q6_k", 1280, 4096, 1, "blocks/q6_k/1"), ("q8_0", 4096, 8192, 6, "strips/q8_0/8"),
    ("q8_0", 4096, 8192, 4, "strips/q8_0/4"), ("q8_0", 16384, 1024, 2, "lines/q8_0/2"), ("q6_k", 6144, 8192, 4, "strips/q6_k/4"),
    ("q6_k", 6144, 511, 2, "quads/q6_k/4"), ("q6_k", 2304, 2304, 1, "strips/q6_k/4"), ("q6_k", 4096, 8192, 1, "spans/q6_k/2"),
    ("q4_k", 4096, 4096, 2, "strips/q4_k/4"), ("q4_k", 2048, 8192, 4, "strips/q4_k/4"), ("q4_k", 2048, 8192, 5, "strips/q4_k/8"),
    ("q4_k", 3840, 4096, 1, "strips/q4_k/4"), ("q4_k", 2560, 5120, 1, "strips/q4_k/4"), ("q4_k", 10240, 16384, 1, "strips/q4_k/4")])
def test_strips_rule(tag, k, rows, m, kernel):
    rng = np.random.default_rng(1821)
    note(f"q8 matvec rule {tag} rows {rows} k {k} m {m}")
    check(tag, "bf16", raw_bytes_for(tag, rng, rows, k), rows, k, rng.normal(0, 1, (m, k) if m > 1 else (k,)).astype(np.float32),
          kernel="gguf_matvec_q8_" + kernel)


def test_strips_activation_rows_in_groups():
    """Eight activation rows of 17408 Q8_0 values do not fit a block's LDS beside its slots: two groups of four."""
    rng = np.random.default_rng(1822)
    rows, k, m = 600, 17408, 8
    weight = hc.TensorDesc.gguf_weight(hc.GgufQuantizedType.kQ8_0, hc.DataType.kFloat32, k, rows)
    assert hc.prepare(context(), Q8, weight, hc.TensorDesc.dense(hc.DataType.kFloat32, [m, k])).dispatch_count() == 2
    note(f"q8 matvec q8_0 [{k} -> {rows}] x {m}: strips, activation rows in groups of four")
    check("q8_0", "f32", weights_for("q8_0", rng, rows, k), rows, k, rng.normal(0, 1.0, (m, k)).astype(np.float32),
          kernel="gguf_matvec_q8_strips/q8_0/4-tokens")


# rows, k, activation rows, how the launch is laid out: sixteen waves to a block, eight where the codes leave no more
# room, or eight where two blocks share a compute unit; a wave to a tile or several ("shared")
FORMS = [(61700, 4352, 4, "16-waves"), (61900, 2304, 8, "16-waves"), (5003, 1792, 4, "16-waves/shared"), (4096, 1280, 5, "16-waves/shared"),
         (66000, 256, 2, "2x8-waves"), (16400, 256, 6, "2x8-waves"), (12289, 1536, 2, "2x8-waves/shared"), (12289, 1536, 6, "2x8-waves/shared")]
EIGHT = {"q4_k": [(520, 35072, 4), (520, 17152, 8)], "q6_k": [(520, 24320, 4), (520, 11776, 8)], "q8_0": [(520, 18176, 4), (520, 8704, 8)]}


@pytest.mark.parametrize("tag", list(KINDS))
def test_strips_every_layout_of_a_launch(tag):
    """The weight repeats 257 distinct rows, so that one meets every place of a tile and of a block: the first 257 products
    are held against the oracle, all others against those, bit by bit (a row's sums do not depend on its place)."""
    rng = np.random.default_rng(1824)
    kind, gguf = KINDS[tag]
    period = 257
    for rows, k, m, form in FORMS + [shape + ("8-waves",) for shape in EIGHT[tag]]:
        raw = weights_for(tag, rng, period, k)
        x = rng.normal(0, 1, (m, k)).astype(np.float32)
        row_bytes = raw.shape[1]
        storage = torch.empty(2 + rows * row_bytes, dtype=torch.uint8, device=DEVICE)[2:]   # two bytes off: no kernel of whole vectors
        distinct = torch.from_numpy(raw).to(DEVICE)
        storage.view(rows, row_bytes).copy_(distinct.repeat((rows + period - 1) // period, 1)[:rows])
        label = f"gguf_matvec_q8_strips/{tag}/{4 if m <= 4 else 8}-tokens/{form}"
        note(f"q8 matvec {tag} [{k} -> {rows}] x {m}: {label}")
        descs = [hc.TensorDesc.gguf_weight(gguf, hc.DataType.kFloat32, k, rows), hc.TensorDesc.dense(hc.DataType.kFloat32, [m, k])]
        (out,) = run(Q8, storage, torch.from_numpy(x).to(DEVICE), descs=descs)
        assert hc.last_launch_variant() == label, hc.last_launch_variant()
        got = out.cpu().numpy().reshape(m, rows)
        centre, bound = orc.gguf_matvec_q8(kind, raw.reshape(-1), period, k, x)
        assert np.all(np.abs(got[:, :period] - centre.reshape(m, period)) <= bound.reshape(m, period))
        assert np.array_equal(got, np.take(got, np.arange(rows) % period, 1))


# Q4_K products on both sides of the limits: more rows than values below 56000 or 32768 rows, of more than 2048 values up to 80 or 100 M
# products, and two to four activation rows up to 115 or 150 M
@pytest.mark.parametrize("x_tag,k,rows,m,kernel", [
    ("bf16", 2048, 6001, 1, "strips"), ("bf16", 2048, 6000, 1, "strips"), ("f32", 2816, 5633, 1, "strips"), ("f32", 3072, 6145, 1, "strips"),
    ("f16", 3072, 6144, 1, "strips"), ("bf16", 1024, 97656, 1, "tiles"), ("bf16", 1024, 97657, 1, "tiles"), ("f32", 2048, 9000, 2, "strips"),
    ("bf16", 1280, 9000, 4, "strips"), ("f16", 2048, 8999, 3, "strips"), ("bf16", 2048, 89999, 2, "tiles"), ("bf16", 2048, 90000, 2, "tiles"),
    ("bf16", 2048, 2049, 1, "strips"), ("f32", 2048, 2048, 1, "tiles"), ("f16", 1024, 1025, 1, "strips"), ("bf16", 1024, 1024, 1, "tiles"),
    ("bf16", 4096, 4097, 1, "strips"), ("bf16", 4096, 4096, 1, "tiles"), ("bf16", 2048, 32767, 1, "strips"), ("f32", 2048, 32768, 1, "tiles"),
    ("bf16", 1536, 55999, 1, "strips"), ("f16", 1536, 56000, 1, "tiles"), ("f32", 1792, 32768, 1, "tiles"),
    ("bf16", 4096, 19531, 1, "strips"), ("bf16", 4096, 19532, 1, "tiles"), ("bf16", 5120, 19531, 1, "strips"), ("bf16", 5120, 19532, 1, "tiles"),
    ("f32", 2048, 6144, 2, "strips"), ("bf16", 2048, 6143, 3, "strips"), ("f16", 1024, 7000, 4, "strips"), ("bf16", 2048, 6144, 4, "strips"),
    ("bf16", 2048, 56152, 2, "strips"), ("bf16", 2048, 56153, 4, "tiles"), ("bf16", 1280, 117187, 3, "strips"), ("bf16", 1280, 117188, 2, "tiles")])
def test_strips_rule_for_many_rows_of_q4_k(x_tag, k, rows, m, kernel):
    rng = np.random.default_rng(1826)
    raw = np.resize(weights_for("q4_k", rng, min(rows, 2000), k), (rows, k // 256 * 144))
    note(f"q8 matvec rule q4_k rows {rows} k {k} m {m}")
    check("q4_k", x_tag, raw, rows, k, rng.normal(0, 1, (m, k) if m > 1 else (k,)).astype(np.float32), kernel=f"gguf_matvec_q8_{kernel}/q4_k/")


# rows, k, activation rows, two bytes off: numbers of waves to a tile that are no powers of two
SPLITS = [(17408, 5120, 5, 0), (17408, 5120, 3, 2),    # three waves to each of five tiles, one without a place
          (600, 2816, 6, 0), (600, 2816, 2, 2),        # eleven to the only tile
          (21504, 2560, 8, 0), (21504, 2560, 8, 2),    # five to each of three tiles, two rounds, one without a place
          (9472, 1536, 7, 2), (8500, 3328, 6, 0)]      # three of eight waves; five of sixteen


@pytest.mark.parametrize("tag", list(KINDS))
def test_strips_any_number_of_waves_to_a_tile(tag):
    """Held as in the test above: 257 distinct rows against the oracle, their repetitions against them bit by bit."""
    rng = np.random.default_rng(1825)
    kind, gguf = KINDS[tag]
    period = 257
    for rows, k, m, off in SPLITS:
        raw = weights_for(tag, rng, period, k)
        x = rng.normal(0, 1, (m, k)).astype(np.float32)
        row_bytes = raw.shape[1]
        storage = torch.empty(off + rows * row_bytes, dtype=torch.uint8, device=DEVICE)[off:]
        storage.view(rows, row_bytes).copy_(torch.from_numpy(raw).to(DEVICE).repeat((rows + period - 1) // period, 1)[:rows])
        note(f"q8 matvec {tag} [{k} -> {rows}] x {m} off {off}: waves to a tile")
        descs = [hc.TensorDesc.gguf_weight(gguf, hc.DataType.kFloat32, k, rows), hc.TensorDesc.dense(hc.DataType.kFloat32, [m, k])]
        (out,) = run(Q8, storage, torch.from_numpy(x).to(DEVICE), descs=descs)
        got = out.cpu().numpy().reshape(m, rows)
        centre, bound = orc.gguf_matvec_q8(kind, raw.reshape(-1), period, k, x)
        assert np.all(np.abs(got[:, :period] - centre.reshape(m, period)) <= bound.reshape(m, period))
        assert np.array_equal(got, np.take(got, np.arange(rows) % period, 1))


@pytest.mark.parametrize("x_tag", ["f32", "bf16"])
@pytest.mark.parametrize("tag", list(KINDS))
def test_strips_blocks_of_few_waves(tag, x_tag):
    """One tile to a block and few activations: a block has only the waves that walk or quantise, one to fifteen."""
    rng = np.random.default_rng(1830)
    for rows, k, m in ((700, 256, 2), (530, 256, 8), (513, 512, 8), (601, 768, 3), (1027, 1280, 5), (600, 1792, 2), (4100, 1792, 8),
                       (600, 2304, 7), (515, 2816, 4), (5200, 1024, 2), (520, 3840, 3), (9300, 768, 4)):
        raw = raw_bytes_for(tag, rng, rows, k)
        for byte_offset in (0, 2):
            note(f"q8 matvec strips few waves {tag} x {x_tag} rows {rows} k {k} m {m} off {byte_offset}")
            check(tag, x_tag, raw, rows, k, rng.normal(0, 1.5, (m, k)).astype(np.float32), byte_offset=byte_offset)
        assert hc.last_launch_variant().startswith(f"gguf_matvec_q8_strips/{tag}/{4 if m <= 4 else 8}-tokens")   # two bytes off: no kernel of whole vectors


@pytest.mark.parametrize("tag,k,rows,m,byte_offset", [
    ("q8_0", 5120, 2304, 6, 0), ("q8_0", 2560, 8192, 4, 0), ("q6_k", 5120, 3584, 8, 0), ("q6_k", 1024, 8192, 5, 0),
    ("q4_k", 4096, 6656, 4, 0), ("q4_k", 9984, 3072, 5, 2)])
def test_strips_are_no_further_from_64_bit_sums(tag, k, rows, m, byte_offset):
    """f32 products of the strip kernel against those of the kernels that serve the same rows in slices of 256 (too
    few for strips), both against the oracle's float64 sums over the same 8-bit codes: the strips' error must not be
    the larger one, over all products (2-norm; summed in 32 bits it was for all of these but the second Q6_K, by 1.04 to 1.2).
    The Q4_K tiles sum in 64 bits too and differ by how many waves share a tile: below, what two roundings leave."""
    rng = np.random.default_rng(1823)
    raw = weights_for(tag, rng, rows, k)
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    kind, gguf = KINDS[tag]
    storage = torch.from_numpy(np.concatenate([np.zeros(byte_offset, np.uint8), raw.reshape(-1)])).to(DEVICE)[byte_offset:].view(rows, -1)
    activations = torch.from_numpy(x).to(DEVICE)

    def products(first, count):
        descs = [hc.TensorDesc.gguf_weight(gguf, hc.DataType.kFloat32, k, count), hc.TensorDesc.dense(hc.DataType.kFloat32, [m, k])]
        (out,) = run(Q8, storage[first:first + count], activations, descs=descs)
        return out.cpu().numpy().astype(np.float64), hc.last_launch_variant()

    note(f"q8 matvec {tag} [{k} -> {rows}] x {m} off {byte_offset}: strips and slices of 256 rows against float64")
    whole, label = products(0, rows)
    assert label.startswith("gguf_matvec_q8_strips"), label
    slices = [products(first, 256) for first in range(0, rows, 256)]
    assert all("strips" not in label for _, label in slices)
    centre, _ = orc.gguf_matvec_q8(kind, raw.reshape(-1), rows, k, x)
    centre = centre.reshape(m, rows)
    own, others = np.linalg.norm(whole - centre), np.linalg.norm(np.concatenate([part for part, _ in slices], 1) - centre)
    twice = np.sqrt(2 / 3) * 2.0 ** -24 * np.linalg.norm(centre)   # test_strips_round_a_product_twice
    assert own <= (max(others, twice) if "tiles" in slices[0][1] else others), f"{own / others:.3f} of the error of the kernels for few rows"


@pytest.mark.parametrize("tag,k,rows,m", [
    ("q4_k", 4352, 1280, 1), ("q4_k", 2560, 12544, 1), ("q4_k", 2304, 12800, 3), ("q6_k", 1792, 2560, 5), ("q6_k", 5632, 3072, 1),
    ("q8_0", 3328, 4352, 8), ("q8_0", 5120, 4608, 5)])
def test_strips_round_a_product_twice(tag, k, rows, m):
    """f32 products against the oracle's float64 sums over the same 8-bit codes.  A product is the sum in 64 bits of its waves'
    shares, each rounded to f32 but the first, and is rounded once itself.  A rounding moves a value by 2^-24 / sqrt(3) of it
    in root mean square, at the foot of a binade, and the shares' squares add up to the product's in the mean: sqrt(2 / 3) * 2^-24 =
    4.9e-8 of the products (2-norm) at most.  (With the lanes' sums rounded first 5.2e-8 to 6.9e-8 at these sizes.)"""
    rng = np.random.default_rng(1827)
    raw = weights_for(tag, rng, rows, k)
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    kind, gguf = KINDS[tag]
    note(f"q8 matvec {tag} [{k} -> {rows}] x {m}: strips against float64")
    descs = [hc.TensorDesc.gguf_weight(gguf, hc.DataType.kFloat32, k, rows), hc.TensorDesc.dense(hc.DataType.kFloat32, [m, k])]
    (out,) = run(Q8, torch.from_numpy(raw.reshape(-1)).to(DEVICE), torch.from_numpy(x).to(DEVICE), descs=descs)
    assert hc.last_launch_variant().startswith("gguf_matvec_q8_strips"), hc.last_launch_variant()
    centre, _ = orc.gguf_matvec_q8(kind, raw.reshape(-1), rows, k, x)
    off = np.linalg.norm(out.cpu().numpy().astype(np.float64).reshape(m, rows) - centre.reshape(m, rows)) / np.linalg.norm(centre)
    assert off <= np.sqrt(2 / 3) * 2.0 ** -24, f"{off:.3e}"


@pytest.mark.parametrize("k,rows,m", [(1024, 500, 1), (2048, 2048, 1), (6144, 300, 1), (8192, 1500, 1), (2048, 32769, 1), (4096, 400, 3), (1280, 511, 8),
                                     (2048, 57000, 2)])
def test_tiles_round_a_product_twice(k, rows, m):
    """The same of the tile kernel, whose waves share a tile by two or four.  (Closed and summed in 32 bits 6.1e-8 to 8.0e-8.)"""
    rng = np.random.default_rng(1831)
    raw = np.resize(weights_for("q4_k", rng, min(rows, 2500), k), (rows, k // 256 * 144))
    x = rng.normal(0, 1, (m, k) if m > 1 else (k,)).astype(np.float32)
    kind, gguf = KINDS["q4_k"]
    note(f"q8 matvec q4_k [{k} -> {rows}] x {m}: tiles against float64")
    descs = [hc.TensorDesc.gguf_weight(gguf, hc.DataType.kFloat32, k, rows), hc.TensorDesc.dense(hc.DataType.kFloat32, list(x.shape))]
    (out,) = run(Q8, torch.from_numpy(raw.reshape(-1)).to(DEVICE), torch.from_numpy(x).to(DEVICE), descs=descs)
    assert hc.last_launch_variant().startswith("gguf_matvec_q8_tiles"), hc.last_launch_variant()
    few = min(rows, 2500)
    centre, _ = orc.gguf_matvec_q8(kind, raw[:few].reshape(-1), few, k, x)
    centre, got = centre.reshape(m, few), out.cpu().numpy().astype(np.float64).reshape(m, rows)[:, :few]
    off = np.linalg.norm(got - centre) / np.linalg.norm(centre)
    assert off <= np.sqrt(2 / 3) * 2.0 ** -24, f"{off:.3e}"


@pytest.mark.parametrize("tag", list(KINDS))
def test_strips_activations_that_are_no_numbers(tag):
    """A NaN is no candidate for a block's magnitude and has the code of a zero; an infinity leaves its block no finite
    scale, so that its activation row's products are NaN; a magnitude whose inverse is none saturates the codes.  In every
    case as in the kernels that serve few rows, and the other activation rows keep their bits."""
    rng = np.random.default_rng(1825)
    kind, gguf = KINDS[tag]
    rows, k, m = 4352, 1280, 6
    raw = weights_for(tag, rng, rows, k)
    storage = torch.from_numpy(np.concatenate([np.zeros(2, np.uint8), raw.reshape(-1)])).to(DEVICE)[2:].view(rows, -1)

    def products(x, first=0, count=rows):
        descs = [hc.TensorDesc.gguf_weight(gguf, hc.DataType.kFloat32, k, count), hc.TensorDesc.dense(hc.DataType.kFloat32, [m, k])]
        (out,) = run(Q8, storage[first:first + count], torch.from_numpy(x).to(DEVICE), descs=descs)
        return out.cpu().numpy(), hc.last_launch_variant()

    clean = rng.normal(0, 1, (m, k)).astype(np.float32)
    clean[0, [5, 300, 301]] = 0.0
    clean[1, 512:768] = 0.0
    odd = clean.copy()
    odd[0, [5, 300, 301]] = [np.nan, -np.nan, np.nan]
    odd[1, 512:768] = np.nan                  # a block without a number
    odd[2, 700] = np.inf
    odd[3, 256] = -np.inf
    odd[4, 256:512] = rng.normal(0, 1e-40, 256)   # 127 / magnitude overflows
    note(f"q8 matvec strips {tag} [{k} -> {rows}] x {m}: NaN, infinities and subnormals among the activations")
    want, label = products(clean)
    got, _ = products(odd)
    assert label.startswith("gguf_matvec_q8_strips")
    for token in (0, 1, 5):
        assert np.array_equal(got[token], want[token]), token
    assert np.isnan(got[2]).all() and np.isnan(got[3]).all()
    general, label = products(odd, 0, 256)
    assert "strips" not in label
    assert np.array_equal(np.isnan(got[:, :256]), np.isnan(general))
    few = np.abs(np.where(np.isnan(general), 0.0, got[:, :256] - general))
    assert np.all(few <= 1e-5 * np.nanmax(np.abs(general)))   # both are within gamma(K / 4 + 65, 2^-24) of the same sum of terms


@pytest.mark.parametrize("tag", ["q4_k", "q6_k"])
def test_strips_activation_blocks_on_both_sides_of_the_short_form(tag):
    """Magnitudes below 2^-60 and from 2^61 on divide in full: whole waves of such blocks, and blocks that share a
    wave with ordinary ones."""
    rng = np.random.default_rng(1825)
    rows, k = 1030, 4096
    x = rng.normal(0, 1, (4, k)).astype(np.float32)
    x[0] *= np.float32(2.0 ** -70)
    x[1] *= np.repeat(np.float32([2.0 ** -62, 1, 2.0 ** -59, 2.0 ** 20]), k // 4)
    x[2] *= np.repeat(np.float32([2.0 ** 58, 2.0 ** 61, 2.0 ** 64, 2.0 ** 60]), k // 4)
    x[3] *= np.tile(np.repeat(np.float32([2.0 ** -65, 2.0 ** -60]), 256), k // 512)
    note(f"q8 matvec strips {tag}: activation blocks below 2^-60 and above 2^61")
    check(tag, "f32", weights_for(tag, rng, rows, k), rows, k, x, kernel=f"gguf_matvec_q8_strips/{tag}/4-tokens")


@pytest.mark.parametrize("tag,rows,m,kernel", [("q4_k", 89999, 5, "strips/q4_k/8"), ("q4_k", 90000, 5, "tiles/q4_k/8"), ("q6_k", 89999, 2, "strips/q6_k/4"),
                                               ("q6_k", 90000, 2, "quads/q6_k/4")])
def test_strips_rule_for_one_span_of_a_vocabulary(tag, rows, m, kernel):
    rng = np.random.default_rng(1825)
    note(f"q8 matvec rule {tag} rows {rows} k 2048 m {m}")
    check(tag, "bf16", raw_bytes_for(tag, rng, rows, 2048), rows, 2048, rng.normal(0, 1, (m, 2048)).astype(np.float32), kernel="gguf_matvec_q8_" + kernel)


def test_strips_scales_of_activation_blocks_are_exact_quotients():
    """A weight row picks one activation block's largest value, whose code is 127: the product is 127 times the block's
    scale, 1 / (127 / largest) in f32, rounded once.  Among the largest values those whose factor has a mantissa of all
    ones, where a quotient by a corrected reciprocal hangs on the reciprocal itself."""
    blocks, m, rows = 16, 8, 512
    raw = np.zeros((rows, blocks, 210), np.uint8)
    quants = np.full(256, 32)
    quants[5] = 33
    for r in range(rows):
        raw[r, :] = pack_q6_k(np.float16(0), np.ones(16), np.full(256, 32))
        raw[r, r % blocks] = pack_q6_k(np.float16(1), np.ones(16), quants)
    rng = np.random.default_rng(1826)
    for draw in range(4):
        largest = (rng.integers(0, 1 << 23, (m, blocks), dtype=np.uint32) | np.uint32(127 << 23)).view(np.float32)
        largest[:, ::4] = np.nextafter(np.float32(63.5), np.float32(64))        # 127 / largest is 2 - 2^-23
        largest *= np.float32(2) ** rng.integers(-59, 50, (m, blocks)).astype(np.float32)
        largest *= rng.choice(np.float32([-1, 1]), (m, blocks))
        x = np.zeros((m, blocks, 256), np.float32)
        x[:, :, 5], x[:, :, 77] = largest, largest * np.float32(0.5)
        factor = np.float32(-127) / largest
        assert (np.abs(factor[:, ::4]).view(np.uint32) & np.uint32(0x7FFFFF) == np.uint32(0x7FFFFF)).all()
        note(f"q8 matvec strips: scales of activation blocks, draw {draw}")
        descs = [hc.TensorDesc.gguf_weight(KINDS["q6_k"][1], hc.DataType.kFloat32, 256 * blocks, rows),
                 hc.TensorDesc.dense(hc.DataType.kFloat32, [m, 256 * blocks])]
        (out,) = run(Q8, torch.from_numpy(raw.reshape(-1)).to(DEVICE), torch.from_numpy(x.reshape(m, -1)).to(DEVICE), descs=descs)
        assert hc.last_launch_variant().startswith("gguf_matvec_q8_strips/q6_k/8")
        wanted = np.float32(-127) * (np.float32(1) / factor)
        assert np.array_equal(out.cpu().numpy(), np.tile(wanted, (1, rows // blocks)))


@pytest.mark.parametrize("rows,m,kernel", [(90000, 1, "spans/q6_k/1"), (90000, 3, "strips/q6_k/4"), (90001, 4, "strips/q6_k/4")])
def test_strips_rule_for_one_span_of_a_vocabulary_and_three_rows_or_more(rows, m, kernel):
    rng = np.random.default_rng(1829)
    note(f"q8 matvec rule q6_k rows {rows} k 2048 m {m}")
    check("q6_k", "bf16", raw_bytes_for("q6_k", rng, rows, 2048), rows, 2048, rng.normal(0, 1, (m, 2048) if m > 1 else (2048,)).astype(np.float32),
          kernel="gguf_matvec_q8_" + kernel)
