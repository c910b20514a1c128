"""The u64 NTT arithmetic with headroom (2^33 <= q < 2^60; no GPU needed): the
device steps of csrc/ntt_kernels.hpp restated in exact integers, every
intermediate truncated to the word as the kernel truncates it.

shoup_add(x, a, w) leaves out the low x low product of the quotient
a floor(w 2^64 / q) / 2^64, so the quotient may be one too small and x grows by
less than 3q for any 64-bit a; reduce_wide brings any word below 3q with the
quotient floor(hi(x) floor(2^64 / q) / 2^32). Both are checked at the edges of
the modulus range with boundary and random operands, and the ranges of a
forward pass (four stages of 3q from below 4q) and of the inverse's sums must
stay below 16q < 2^64. A planted mistake (the middle sum's carry dropped) fails."""
import random

import pytest

MASK = (1 << 64) - 1
LOW = (1 << 32) - 1


def shoup_add(x, a, w, q, carry=True):
    wp = (w << 64) // q
    al, ah, pl, ph = a & LOW, a >> 32, wp & LOW, wp >> 32
    mid = ah * pl + al * ph
    m1, over = mid & MASK, (mid >> 64) if carry else 0
    quotient = (ah * ph + (m1 >> 32) + (over << 32)) & MASK
    nq = -q & MASK
    p = ((al * (w & LOW) + x) + (quotient & LOW) * (nq & LOW)) & MASK
    k = (al * (w >> 32) + ah * (w & LOW) + (quotient & LOW) * (nq >> 32) + (quotient >> 32) * (nq & LOW)) & LOW
    return (p + (k << 32)) & MASK


def reduce_wide(x, q):
    m = (1 << 64) // q
    assert m < 1 << 32
    k = ((x >> 32) * m) >> 32
    return (x - k * q) & MASK


MODULI = [(1 << 33) + 1, (1 << 33) + (1 << 32) + 3, (1 << 45) - 5, (1 << 59) + 1, 576460756061519873,
          1152921504577486849, (1 << 60) - 1]


def words(rng, q):
    edges = [0, 1, q - 1, q, 2 * q, 3 * q - 1, 16 * q - 1, LOW, 1 << 32, MASK, MASK - 1, (LOW << 32), MASK ^ LOW]
    return [e for e in edges if 0 <= e <= MASK] + [rng.getrandbits(64) for _ in range(300)]


def ok_product(a, w, q, **kw):
    v = shoup_add(0, a, w, q, **kw)
    return v < 3 * q and v % q == a * w % q


@pytest.mark.parametrize("q", MODULI)
def test_products_and_reductions(q):
    rng = random.Random(q)
    ws = [0, 1, 2, q - 1, q - 2, q >> 1] + [rng.randrange(q) for _ in range(60)]
    for a in words(rng, q):
        r = reduce_wide(a, q)
        assert r < 3 * q and r % q == a % q
        for w in ws:
            assert ok_product(a, w, q)
            x = rng.randrange(13 * q)
            y = shoup_add(x, a, w, q)  # x + v, no wrap below 16q
            assert x <= y < x + 3 * q and y % q == (x + a * w) % q
            assert (2 * x + 3 * q - y) & MASK < 16 * q  # the butterfly's other output


def test_dropped_carry_fails():
    q = MODULI[-1]
    rng = random.Random(1)
    cases = [(a, rng.randrange(q)) for a in words(rng, q) for _ in range(40)]
    assert all(ok_product(a, w, q) for a, w in cases)
    assert not all(ok_product(a, w, q, carry=False) for a, w in cases)


@pytest.mark.parametrize("lengths", [(lt,) for lt in range(1, 15)] + [(l1, l2) for l1 in range(4, 10) for l2 in range(4, 13)])
def test_forward_ranges(lengths):
    """A phase reduces its values where its stages would pass 16q."""
    bound = 4
    for lt in lengths:
        done = 0
        while done < lt:
            stages = min(4, lt - done)
            if bound + 3 * stages > 16:
                bound = 3
            bound += 3 * stages
            assert bound <= 16
            done += stages


def test_inverse_ranges():
    """Sums double, products are below 3q, and a pair whose sum would pass 16q
    is reduced first; both sides of a pair always share one of 3, 6 or 12."""
    bound = [3] * 16
    for bit in range(4):
        for r in range(16):
            if r >> bit & 1:
                continue
            r2 = r | 1 << bit
            assert bound[r] == bound[r2] and bound[r] in (3, 6, 12)
            if bound[r] + bound[r2] > 16:
                bound[r] = bound[r2] = 3
            bound[r], bound[r2] = bound[r] + bound[r2], 3
            assert bound[r] <= 16
