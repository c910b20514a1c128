"""The u64 NTT arithmetic with headroom (2^33 <= q < 2^60; no GPU needed): the
device steps of csrc/ntt_kernels.hpp restated in exact integers, every
intermediate truncated to the word as the kernel truncates it.

shoup_add(x, a, w) leaves out the low x low product of the quotient
a floor(w 2^64 / q) / 2^64, so the quotient may be one too small and x grows by
less than 3q for any 64-bit a; reduce_wide brings any word below 3q with the
quotient floor(hi(x) floor(2^64 / q) / 2^32). Both are checked at the edges of
the modulus range with boundary and random operands. Where the kernels reduce is
read from their own schedule, csrc/ntt_schedule.hpp compiled for the host: every
pass's ranges must stay below 16q < 2^64. Planted mistakes (the middle sum's
carry dropped, a higher limit, a reduction left out) fail."""
import random
import subprocess
from pathlib import Path

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


# ---- the kernels' own schedule ------------------------------------------------

SCHEDULE = Path(__file__).resolve().parent.parent / "cubutterfly_amd" / "csrc" / "ntt_schedule.hpp"

PROGRAM = r"""
#include "ntt_schedule.hpp"
#include <cstdio>
using namespace cbw::ntt_detail;
int main() {
    std::printf("E %d\n", kHeadroomEntry);
    for (int lt = 1; lt <= 14; ++lt) {
        for (int entry = 3; entry <= 16; ++entry) {
            std::printf("X %d %d %d\n", lt, entry, forward_exit(lt, entry));
            for (int p = 0; p < num_phases(lt); ++p)
                std::printf("F %d %d %d %d\n", lt, entry, p, int(forward_reduces(lt, p, entry)));
        }
        for (int ct = 0; ct < 2; ++ct)
            for (int p = 0; p < num_phases(lt); ++p)
                for (int s = 0; s < active_stages(lt, ct, p); ++s)
                    std::printf("S %d %d %d %d %d\n", lt, ct, p, exec_stage(lt, ct, p, s), window_start(lt, ct, p));
        for (int last = 0; last < 2; ++last)
            for (int p = 0; p < num_phases(lt); ++p) {
                const InversePhase ph = inverse_phase(lt, p, last);
                for (int s = 0; s < active_stages(lt, false, p); ++s)
                    for (int r = 0; r < kE; ++r)
                        std::printf("I %d %d %d %d %d %d %d\n", lt, last, p, s, r, int(ph.reduce[s][r]), ph.enter[s][r]);
                for (int r = 0; r < kE; ++r) std::printf("L %d %d %d %d %d\n", lt, last, p, r, int(ph.reduce_last[r]));
            }
    }
}
"""


def read_schedule(folder, header):
    """The header's functions, compiled and printed: rows of whole numbers by letter."""
    (folder / "ntt_schedule.hpp").write_text(header)
    (folder / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", str(folder), str(folder / "main.cpp"), "-o", str(folder / "main")],
                   check=True)
    out = subprocess.run([str(folder / "main")], check=True, capture_output=True, text=True).stdout
    rows = {}
    for line in out.splitlines():
        letter, *numbers = line.split()
        rows.setdefault(letter, []).append(tuple(map(int, numbers)))
    return rows


def check_schedule(rows):
    """Walks every pass with the printed decisions alone: values as upper bounds in
    units of q, all below 16q < 2^64, each transform bit butterflied once."""
    entry = rows["E"][0][0]
    assert entry >= 3  # reduced input words are below 3q
    stages = {}
    for lt, ct, p, k, ws in rows["S"]:
        stages.setdefault((lt, ct), []).append((p, k, k - ws))
    reduces = {(lt, b, p): r for lt, b, p, r in rows["F"]}
    exits = {(lt, b): x for lt, b, x in rows["X"]}
    enter = {row[:5]: row[5:] for row in rows["I"]}
    last = {row[:4]: row[4] for row in rows["L"]}

    def forward(lt, bound):
        phase = -1
        for p, k, jb in stages[lt, 1]:
            assert 0 <= jb < 4
            if p != phase and reduces[lt, bound_in, p]:
                bound = 3
            phase = p
            bound += 3  # x + v and x + 3q - v, v below 3q
            assert bound <= 16, (lt, bound_in, p)
        return bound

    for lt in range(1, 15):
        for ct in (0, 1):
            assert sorted(k for _, k, _ in stages[lt, ct]) == list(range(lt))
        bound_in = entry  # one-pass rows and column passes
        assert exits[lt, entry] == forward(lt, entry)
        for l1 in range(4, 10):  # row passes take what a column pass of 2^l1 points leaves
            bound_in = exits[l1, entry]
            assert exits[lt, bound_in] == forward(lt, bound_in)
        for final in (0, 1):
            for p in range((lt + 3) // 4):
                bound = [3] * 16
                done = [(k, jb) for q, k, jb in stages[lt, 0] if q == p]
                for s, (k, jb) in enumerate(done):
                    for r in range(16):
                        if r >> jb & 1:
                            continue
                        r2 = r | 1 << jb
                        assert enter[lt, final, p, s, r][0] == enter[lt, final, p, s, r2][0]
                        if enter[lt, final, p, s, r][0]:
                            bound[r] = bound[r2] = 3
                        span = 3 if enter[lt, final, p, s, r2][1] <= 3 else 6
                        assert span >= bound[r2] and bound[r] + span <= 16 and bound[r] + bound[r2] <= 16
                        scaled = final and k == lt - 1
                        bound[r], bound[r2] = 3 if scaled else bound[r] + bound[r2], 3
                assert all(b <= 3 or last[lt, final, p, r] for r, b in enumerate(bound))


def test_schedule_stays_in_range(tmp_path):
    check_schedule(read_schedule(tmp_path, SCHEDULE.read_text()))


@pytest.mark.parametrize("planted", [("kHeadroomLimit = 16", "kHeadroomLimit = 24"), ("kHeadroomEntry = 4", "kHeadroomEntry = 1"),
                                     ("ph.reduce_last[r] = bound[r] > kReduced", "ph.reduce_last[r] = bound[r] > 6")])
def test_planted_range_mistakes_fail(tmp_path, planted):
    text = SCHEDULE.read_text()
    assert planted[0] in text
    rows = read_schedule(tmp_path, text.replace(*planted))
    with pytest.raises(AssertionError):
        check_schedule(rows)
