"""The identities the packed aggregation search relies on, checked on the CPU over
all their forms: the part of a full-size node's key for every 16-bit hash and every
leaf size's two levels, the slot arithmetic that shares the fold's first multiply
between eight consecutive candidates, and the node sizes the state's bounds hold."""
import numpy as np
import pytest

M32 = np.uint64(0xFFFFFFFF)
C1 = 0x85EBCA6B


def _levels(leaf):
    lower = leaf * max(2, -(-(35 * leaf + 50) // 100))
    upper = lower * (2 if leaf < 7 else -(-(21 * leaf + 90) // 100))
    return [(leaf, lower), (lower, upper)]


@pytest.mark.parametrize("leaf", range(2, 25))
def test_part_is_one_high_multiply(leaf):
    h = np.arange(65536, dtype=np.uint64)
    for unit, m in _levels(leaf):
        fan = m // unit
        assert fan * unit == m and fan <= 9 and m < 4096
        want = ((h * np.uint64(m)) >> np.uint64(16)) // np.uint64(unit)
        got = (h * np.uint64(fan << 16)) >> np.uint64(32)  # 24-bit operands, upper half of the product
        assert np.array_equal(want, got)
        assert int(got.max()) == fan - 1


def test_slots_share_the_first_multiply():
    rng = np.random.default_rng(5)
    lane8 = np.arange(64, dtype=np.uint64) * np.uint64(8)
    for r in range(8):
        for _ in range(300):
            lo = (int(rng.integers(0, 1 << 29)) << 3 | r) & 0xFFFFFFFF
            hi = int(rng.integers(0, 1 << 32))
            if (lo & 0xFFFF) > 0xFFFF - (8 * 64 + 8):
                continue
            D = hi ^ (hi >> 16) ^ (lo >> 16)
            q = [(((np.uint64((lo - r + 8 * k) & 0xFFFFFFFF) + lane8) ^ np.uint64(D)) * np.uint64(C1)) & M32
                 for k in range(2)]
            s = [(-(C1 << b) if D >> b & 1 else C1 << b) for b in range(3)]
            for u in range(8):
                j = (r + u) & 7
                sj = sum(s[b] for b in range(3) if j >> b & 1) & 0xFFFFFFFF
                got = (q[(r + u) >> 3] + np.uint64(sj)) & M32
                w = np.uint64(lo) + lane8 + np.uint64(u)  # no carry into the high word here
                t = w ^ np.uint64(hi)
                t = t ^ (t >> np.uint64(16))
                assert np.array_equal(got, (t * np.uint64(C1)) & M32)
