"""The derivation of the device FNV-1a's four-bit levels and of its sums on the matrix cores, restated on the CPU and compared
with the byte loop.  These are checks of the mathematics: the kernel's own functions and tables are compiled and compared
with the byte loop in tests/test_hash_math.py."""
import numpy as np
import pytest

P, MASK = 1099511628211, (1 << 64) - 1
LOW = P & 0xFF
INV_LOW = pow(LOW, -1, 1 << 64)


def run(l, data):
    for b in data:
        l = ((l ^ int(b)) * LOW) & 0xFF
    return l


def map_of(low, j, k, data):
    """2^(k-2) machines, the top bit's terms for a set bit below it from the byte parities."""
    ends = [run(low | (m << j), data) for m in range(1 << (k - 2))]
    flip = ((int(np.bitwise_xor.reduce(data)) if len(data) else 0) >> (j + k - 2) & 1) ^ (len(data) & 1)
    out = 0
    for i in range(k):
        for at in range(1 << i):
            e = ends[sum(((at >> (i - 1 - b)) & 1) << b for b in range(min(i, k - 2)))]
            term = (e >> (j + i)) & 1
            if i == k - 1 and at & 1:
                term ^= ((e >> (j + k - 2)) & 1) ^ flip
            out |= term << ((1 << i) - 1 + at)
    return out


def apply(k, m, st):
    out, at = st, 0
    for i in range(k):
        out ^= ((m >> ((1 << i) - 1 + at)) & 1) << i
        at = 2 * at + ((st >> i) & 1)
    return out


def compose(k, g, f, i=0, at=0, gat=0):
    base, nxt = (1 << i) - 1, (2 << i) - 1
    t = (f >> (base + at)) & 1
    r = (t ^ ((g >> (base + gat)) & 1)) << (base + at)
    if i + 2 == k:
        pair = (g >> (nxt + 2 * gat)) & 3
        if t:
            pair = (pair >> 1) | ((pair & 1) << 1)
        return r | ((((f >> (nxt + 2 * at)) & 3) ^ pair) << (nxt + 2 * at))
    return r | compose(k, g, f, i + 1, 2 * at, 2 * gat + t) | compose(k, g, f, i + 1, 2 * at + 1, 2 * gat + (t ^ 1))


@pytest.mark.parametrize("j,k", [(0, 4), (4, 4), (0, 3), (3, 3), (6, 2)])
def test_level_maps_take_every_start_to_its_end(j, k):
    rng = np.random.default_rng(17 + 8 * j + k)
    for trial in range(200):
        data = rng.integers(0, 256, int(rng.integers(0, 200)))
        if trial % 3 == 0:
            data &= int(rng.integers(0, 256))
        low = int(rng.integers(0, 256)) & ((1 << j) - 1)
        cut = int(rng.integers(0, len(data) + 1))
        whole = map_of(low, j, k, data)
        first, second = map_of(low, j, k, data[:cut]), map_of(run(low, data[:cut]) & ((1 << j) - 1), j, k, data[cut:])
        assert compose(k, second, first) == whole
        for st in range(1 << k):
            assert apply(k, whole, st) == (run(low | (st << j), data) >> j) & ((1 << k) - 1)


def test_wave_maps_by_counting_lower_lanes():
    """64 lanes' maps from a start state, each bit by the parity of the lower lanes' terms."""
    rng = np.random.default_rng(3)
    for k in (2, 3, 4):
        for st in range(1 << k):
            maps = [int(x) for x in rng.integers(0, 1 << ((1 << k) - 1), 64)]
            want, s = [], st
            for m in maps:
                want.append(s)
                s = apply(k, m, s)
            at, bits, end = [0] * 64, [0] * 64, st
            for i in range(k):
                terms = [(m >> ((1 << i) - 1 + a)) & 1 for m, a in zip(maps, at)]
                low = [(sum(terms[:l]) & 1) ^ ((st >> i) & 1) for l in range(64)]
                end ^= (sum(terms) & 1) << i
                bits = [b | (x << i) for b, x in zip(bits, low)]
                at = [2 * a + x for a, x in zip(at, low)]
            assert bits == want and end == s


def digits(v):
    out = []
    for _ in range(8):
        d = v & 0xFF
        d -= 256 if d >= 128 else 0
        out.append(d)
        v = ((v - d) & MASK) >> 8
    return out


def test_matrix_sum_of_a_wave_equals_the_byte_loop():
    """16 KiB as 64 segments of two 128-byte halves: the products' offset bytes times the signed digits of the weights,
    rows of lanes 16 apart summed together, exact in 32 bits, give the wave's part of the hash."""
    rng = np.random.default_rng(9)
    data = rng.integers(0, 256, 16384)
    h0 = int(rng.integers(0, 1 << 63))
    state = [h0 & 0xFF]
    for b in data:
        state.append(((state[-1] ^ int(b)) * LOW) & 0xFF)
    prod = np.array([LOW * (l ^ int(b)) for l, b in zip(state, data)]).reshape(4, 16, 2, 128)   # [group][row][half][byte]
    lo, hi = (prod & 0xFF) - 128, (prod >> 8) - 128
    p_inv = pow(P, -1, 1 << 64)

    def weights(pe):   # of a product's low and high byte
        return (INV_LOW * pe - p_inv * pe) & MASK, (256 * INV_LOW * pe) & MASK

    w = np.zeros((4, 2, 128, 2, 8), dtype=np.int64)
    offset = 0
    for q in range(4):
        for half in range(2):
            for c in range(128):
                pe = pow(P, 256 - 128 * half - c, 1 << 64)
                pair = weights(pe * pow(P, 4096 * (3 - q), 1 << 64) & MASK)
                w[q, half, c] = [digits(x) for x in pair]
                if q == 0:
                    offset += sum(weights(pe))
    sums = np.einsum("qrhc,qhcd->rd", lo, w[..., 0, :]) + np.einsum("qrhc,qhcd->rd", hi, w[..., 1, :])
    assert np.abs(w).max() <= 128 and np.abs(sums).max() < 1 << 31
    total = sum(int(sums[r, d]) * (1 << (8 * d)) * pow(P, 256 * (15 - r), 1 << 64) for r in range(16) for d in range(8))
    for lane in range(64):
        ends = state[256 * lane + 256] - state[256 * lane] * pow(P, 256, 1 << 64) + 128 * offset
        total += ends * pow(P, 256 * (63 - lane), 1 << 64)
    h = h0
    for b in data:
        h = ((h ^ int(b)) * P) & MASK
    assert (h0 * pow(P, 16384, 1 << 64) + total) & MASK == h
