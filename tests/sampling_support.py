"""Independent forms for the sampling tests: Philox4x32-10 over numpy arrays (the equations of
Random123's philox4x32_10 as the reference's fixture restates them, tests/compute_models/
sampling_fixture.h:70-91), the fixture's identities and logits (…:93-101,214-223) and the float64
inverse CDF of a row's uniform with the band of indices rounding can move the answer within."""
from __future__ import annotations

import numpy as np

from oracle import lib as orc


def philox_array(counters: np.ndarray, keys: np.ndarray) -> np.ndarray:
    """counters [n, 4], keys [n, 2] (uint32) -> [n, 4] words."""
    c = [counters[:, i].astype(np.uint64) for i in range(4)]
    k = [keys[:, i].astype(np.uint64) for i in range(2)]
    mask = np.uint64(0xFFFFFFFF)
    for _ in range(10):
        p0 = c[0] * np.uint64(0xD2511F53)
        p1 = c[2] * np.uint64(0xCD9E8D57)
        c = [((p1 >> np.uint64(32)) ^ c[1] ^ k[0]) & mask, p1 & mask, ((p0 >> np.uint64(32)) ^ c[3] ^ k[1]) & mask, p0 & mask]
        k = [(k[0] + np.uint64(0x9E3779B9)) & mask, (k[1] + np.uint64(0xBB67AE85)) & mask]
    return np.stack(c, axis=1).astype(np.uint32)


def fixture_identities(rows: int, draw: int) -> np.ndarray:
    r = np.arange(rows, dtype=np.uint64)
    with np.errstate(over="ignore"):
        draws = np.uint64(draw) + r
    out = np.stack([(r * np.uint64(0x9E3779B9)) & np.uint64(0xFFFFFFFF),
                    np.uint64(0xFEDCBA98) ^ ((r * np.uint64(17)) & np.uint64(0xFFFFFFFF)),
                    draws & np.uint64(0xFFFFFFFF), draws >> np.uint64(32)], axis=1)
    return out.astype(np.uint32).reshape(rows, 4)


def fixture_logits(rows: int, width: int, type_id: int):
    """(storage, float32 values after the storage's rounding)."""
    r, j = np.meshgrid(np.arange(rows), np.arange(width), indexing="ij")
    values = (((r * 7 + j) % 11 - 5) * 0.25 + np.where(r % 3 == 0, 1024.0, -1024.0)).astype(np.float32)
    values[j % 5 == 0] = -np.inf
    if type_id == orc.F32:
        return values, values
    stored = orc.from_f32(type_id, values)
    return stored, orc.to_f32(type_id, stored)


def uniform_of(words) -> float:
    return (float(words[0]) * 2.0 ** 20 + float(int(words[1]) >> 12) + 0.5) * 2.0 ** -52


def inverse_cdf_bounds(values: np.ndarray, identities: np.ndarray, slack: float = 4e-6):
    """Per row the lowest and highest index an inverse-CDF draw of the row's uniform may return
    when every mass carries a relative error of up to `slack`, and the float64 log probability of
    every element.  values: float32 [rows, width] (the logical log-weights)."""
    rows, width = values.shape
    v = values.astype(np.float64)
    maximum = v.max(axis=1, keepdims=True)
    mass = np.exp(v - maximum)
    total = mass.sum(axis=1)
    scores = (v - maximum) - np.log(total)[:, None]
    cumulative = np.cumsum(mass, axis=1)
    low, high = np.zeros(rows, np.int64), np.zeros(rows, np.int64)
    for r in range(rows):
        block = philox_array(np.array([[0, 0, identities[r, 2], identities[r, 3]]], np.uint32),
                             np.array([identities[r, :2]], np.uint32))[0]
        threshold = total[r] * uniform_of(block)
        band = slack * total[r]
        positive = np.nonzero(mass[r] > 0)[0]
        first = np.searchsorted(cumulative[r], threshold - band, side="right")
        last = np.searchsorted(cumulative[r], threshold + band, side="right")
        # an index without mass is never returned: move to the neighbours that have some
        low[r] = positive[np.searchsorted(positive, min(first, width - 1), side="left").clip(0, positive.size - 1)]
        high[r] = positive[np.searchsorted(positive, min(last, width - 1), side="left").clip(0, positive.size - 1)]
    return low, high, scores


def running_sums(masses: np.ndarray) -> np.ndarray:
    """[rows, lanes] f64 -> what each lane holds after a scan that adds the sum 1, 2, 4, ... lanes below."""
    through = masses.astype(np.float64).copy()
    step = 1
    while step < through.shape[1]:
        through[:, step:] = through[:, step:] + through[:, :-step].copy()
        step *= 2
    return through


def rows_with_a_threshold_between_sums(mass_of, identities: np.ndarray, seed: int):
    """float32 logits [n, 256] and their identities whose threshold falls where the running sums of sixteen elements
    a lane are not monotone: lane 7 has no mass (-inf), its own sum is above lane 6's by the last bit, and the threshold
    lies from lane 6's sum to below lane 7's.  `mass_of(float32 array)`: the kernel's exp of values up to 0, as float32.
    Only the rows for which the arithmetic lands there; the last element in front of lane 7 has no mass either."""
    rng = np.random.default_rng(seed)
    rows, lanes, hole = identities.shape[0], 16, 7
    words = philox_array(np.stack([np.zeros(rows, np.uint32)] * 2 + [identities[:, 2], identities[:, 3]], axis=1), identities[:, :2])
    uniform = np.array([uniform_of(w) for w in words])
    t = np.full((rows, lanes, 16), -np.inf, np.float32)
    t[:, :hole] = -rng.uniform(0, 5, (rows, hole, 16)) ** 2  # so far apart that sums round
    t[:, 0, 0], t[:, hole - 1, 15] = 0, -np.inf
    lane_mass = lambda: np.add.accumulate(mass_of(t).astype(np.float64), axis=2)[:, :, -1]
    front = running_sums(lane_mass())[:, hole - 1]
    # what lies behind the hole: bulk, then ever smaller masses that close what is left of the wanted sum
    wanted = front / uniform - front
    place = (hole + 1) * 16
    flat = t.reshape(rows, 256)
    for _ in range(256 - place - 8):
        bulk = wanted > 1.0
        flat[bulk, place] = np.float32(-0.1)
        wanted[bulk] -= mass_of(flat[bulk, place]).astype(np.float64)
        place += 1
    for _ in range(8):
        start = np.log(np.maximum(wanted, 1e-300)).astype(np.float32)
        steps = np.arange(-8, 9, dtype=np.int64)[None, :]
        near = (start.view(np.int32).astype(np.int64)[:, None] + steps).astype(np.int32).view(np.float32)
        masses = mass_of(near).astype(np.float64)
        masses[~((near < 0) & (near > -60) & (masses <= wanted[:, None]))] = -1.0
        best = masses.argmax(axis=1)
        found = masses[np.arange(rows), best] > 0
        flat[found, place] = near[np.arange(rows), best][found]
        wanted[found] -= masses[np.arange(rows), best][found]
        place += 1
    # the row's total as the kernel takes it: four elements a lane, then pairs 1, 2, 4, ... lanes apart
    total = np.add.accumulate(mass_of(flat).astype(np.float64).reshape(rows, 64, 4), axis=2)[:, :, -1]
    while total.shape[1] > 1:
        total = total[:, 0::2] + total[:, 1::2]
    threshold = total[:, 0] * uniform
    through = running_sums(lane_mass())
    armed = (through[:, hole - 1] <= threshold) & (threshold < through[:, hole])
    return flat[armed], identities[armed]
