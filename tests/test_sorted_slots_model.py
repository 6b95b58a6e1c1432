"""The doubles by which the KNN kernels keep MinK's slots as a sorted list, against the oracle.

`knn_filter_kernel_f32` (4 to 32 slots, a query per lane) and `knn_wave_kernel_f32` (64 slots, a query per wave) in
torkit3d_amd/csrc/knn.hip do not keep a query's k distances in slot order as the reference's MinK does
(csrc/include/mink.cuh:61-89) but in descending order, each as a double: the bits of the distance above a flag, the
number of slots less one less the slot, and the key (`KnnSlot`). An insertion is a minimum and a maximum per position. This
file restates that on 64-bit patterns and checks it against the CPU oracle's literal MinK on sequences where equal
distances are everywhere, which is where the slot order shows, with zeros, subnormal and infinite distances, NaNs and
the largest keys that a slot has bits for. It runs without a GPU; the kernels themselves are checked against the oracle
by tests/test_gpu_knn.py and tests/test_gpu_knn_wave.py.
"""
import math
import random

import numpy as np
import pytest

import oracle

NAN_OF_THE_FILL, NOT_INSERTED, UNUSED = 0xff800000, 0x7fe00000, -math.inf


class Slots:
    """The low word's fields, as KnnSlot<kmax> has them."""

    def __init__(self, kmax):
        self.kmax, self.key_bits = kmax, 31 - int(math.log2(kmax))
        self.flag, self.slot_mask = 1 << 31, (kmax - 1) << self.key_bits

    def pack(self, high, low):
        return np.array([high << 32 | low], np.uint64).view(np.float64)[0]

    def first(self, high, slot):  # key `slot` in slot `slot`, as the fill leaves it
        return self.pack(high, (self.kmax - 1 - slot) << self.key_bits | slot)

    def unpack(self, v):
        """(bits of the distance, low word, slot, key) of a position."""
        word = int(np.array([v]).view(np.uint64)[0])
        low = word & 0xffffffff
        return word >> 32, low, self.kmax - 1 - ((low & self.slot_mask) >> self.key_bits), low & ((1 << self.key_bits) - 1)


def sink(v, x):
    """The chain of an insertion: the head leaves, x goes to its place."""
    below = np.append(v[1:], UNUSED)
    return np.maximum(below, np.minimum(v, x))


def ordered_by_network(v, k):
    """The first k lanes in descending order, by the steps of knn_order_lanes."""
    steps = [(1, [1]), (2, [3, 1]), (4, [7, 2, 1]), (8, [15, 4, 2, 1]), (16, [31, 8, 4, 2, 1]), (32, [63, 16, 8, 4, 2, 1])]
    lane = np.arange(64)
    for least, xors in steps:
        for x in xors if k > least else []:
            other = v[lane ^ x]
            lower = lane < (lane ^ x)
            v = np.where((other > v) == lower, other, v)
    return v


def bits_of(dist):
    return [int(b) for b in np.asarray(dist, np.float32).view(np.uint32)]


def doubles_knn(dist, k, kmax, wave, key_of, long=False):
    """MinK's (distance bits, keys) in slot order for one query. `key_of`: the number a key beyond the fill has. `long`:
    the numbers beside the slots instead of in them."""
    s, bits = Slots(kmax), bits_of(dist)
    high = [NAN_OF_THE_FILL if d != d else b for d, b in zip(dist[:k], bits)]
    v = np.full(kmax, UNUSED)
    if wave:
        v[:k] = [s.first(h, i) for i, h in enumerate(high)]
        v = ordered_by_network(v, k)
    else:
        for i, h in enumerate(high):
            x = s.first(h, i)
            for p in range(i, 0, -1):
                v[p] = max(v[p], min(v[p - 1], x))
            v[0] = max(v[0], x)
    number = np.array([s.unpack(a)[2] for a in v])
    frozen = dist[0] != dist[0]
    for j in range(k, len(dist)):
        top, low, slot, _ = s.unpack(v[0])
        maximum = -math.inf if frozen else np.array([top], np.uint32).view(np.float32)[0]
        inserted = bool(dist[j] < maximum)
        if wave and not inserted:
            continue
        flag = s.flag if bits[j] >= s.unpack(v[1])[0] or s.unpack(v[1])[0] >= 1 << 31 else 0
        x = s.pack(bits[j] if inserted else NOT_INSERTED, low & s.slot_mask | flag | (0 if long else key_of(j)))
        after = sink(v, x)
        if long:
            below = np.append(v[1:], UNUSED)
            number = np.where(after == below, np.append(number[1:], 0), np.where(after == v, number, key_of(j)))
        assert inserted or np.array_equal(after.view(np.uint64), v.view(np.uint64))
        v = after
    out_d, out_i = [None] * k, [None] * k
    for p in range(k):
        top, _, slot, key = s.unpack(v[p])
        out_d[slot] = bits[slot] if top == NAN_OF_THE_FILL else top
        out_i[slot] = int(number[p]) if long else key
    return out_d, out_i


def sequence(rnd, k):
    n = max(rnd.choice([k, k + 1, 40, 150, 400]), k)
    levels = rnd.choice([2, 3, 5, 17, 1000])   # distinct coordinates: few = ties everywhere
    scale = rnd.choice([1.0, 1.0, 1e-21, 1e18])  # subnormal distances, some that overflow
    xs = [rnd.randrange(levels) * scale for _ in range(n)]
    if rnd.random() < 0.2:
        xs.sort(reverse=True)                   # far to near: every key is inserted
    if rnd.random() < 0.15:
        for _ in range(3):
            xs[rnd.randrange(min(n, k + 3))] = math.nan
    if rnd.random() < 0.1:
        xs[rnd.randrange(n)] = math.inf
    return xs


FORMS = [(4, False, False), (8, False, False), (16, False, False), (32, False, False), (64, True, False), (64, True, True)]


@pytest.mark.parametrize("kmax,wave,long", FORMS)
def test_sorted_list_rule_reproduces_mink_slot_order(kmax, wave, long):
    rnd = random.Random(kmax)
    least = 1 if kmax in (4, 64) else kmax // 2 + 1
    for trial in range(120):
        k = rnd.randint(least, kmax)
        xs = sequence(rnd, k)
        key = np.zeros((1, len(xs), 3), np.float32)
        key[0, :, 0] = xs
        want_d, want_i = oracle.knn(np.zeros((1, 1, 3), np.float32), key, k)
        with np.errstate(over="ignore", under="ignore"):
            dist = key[0, :, 0] * key[0, :, 0]   # as the oracle forms them
        # keys behind the fill count up to the largest that a slot has bits for, long ones beyond
        shift = ((1 << 29) if long else (1 << (31 - int(math.log2(kmax))))) - len(xs)
        got_d, got_i = doubles_knn(dist, k, kmax, wave, lambda j: j + shift, long)
        want = [int(i) + (shift if i >= k else 0) for i in want_i[0, 0]]
        assert got_i == want, "trial %d" % trial
        got = np.array(got_d, np.uint32).view(np.float32)
        np.testing.assert_array_equal(got, want_d[0, 0], err_msg="trial %d" % trial)


def test_every_pattern_of_a_distance_is_a_finite_double_in_order():
    # zero, the smallest subnormal, the largest finite value, infinity, and a key that is not inserted above them all;
    # below: the NaN of the fill, then unused slots
    s = Slots(64)
    row = [s.first(high, 0) for high in (0, 1, 0x007fffff, 0x7f7fffff, 0x7f800000, NOT_INSERTED)]
    assert all(math.isfinite(v) for v in row) and row == sorted(row)
    for slot in (0, 63):
        assert UNUSED < s.first(NAN_OF_THE_FILL, slot) < row[0]
    # among equal distances: ascending slots, the flag in front
    assert s.first(5, 0) > s.first(5, 1) and s.pack(5, s.flag) > s.first(5, 0)


@pytest.mark.parametrize("k", range(1, 65))
def test_network_orders_the_first_lanes(k):
    rng = np.random.default_rng(k)
    v = np.full(64, UNUSED)
    v[:k] = rng.permutation(64)[:k]
    np.testing.assert_array_equal(ordered_by_network(v, k), np.sort(v)[::-1])
