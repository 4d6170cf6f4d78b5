"""The banded runs of the overlap aligner at the edges of their forms, against
the CPU oracle: block and chunk remainders, every group of lanes (8 to 64, and
256 over the four waves of a team), bands too wide for the lanes of a wave and
of a team (strips), band guesses that must grow, few long pairs (a team of
waves per pair) alone and beside many (one wave per pair), long pairs on one
wave each, long gaps, and target bytes other than A, C, G and T at chunk edges.
"""
import sys

import numpy as np
import pytest

from racon_amd import _lib
from synth import make_pair, mutate, random_seq
from test_zz_no_alloc import Hip, noalloc_align

sys.path.insert(0, _lib.PKG_DIR + "/../oracle")
import oracle_py  # noqa: E402

pytestmark = pytest.mark.gpu


def check(pairs, band=0, only=None, launches=None):
    """launches: 2 for teams beside one wave per pair, 1 for either alone."""
    b = _lib.AlignBatch()
    if band:
        b.set_band(band)
    b.upload(pairs)
    b.run()
    ops, dist = b.download()
    assert launches in (None, b.stats().launches)
    b.close()
    compare(pairs, ops, dist, only)


def compare(pairs, ops, dist, only=None):
    for i, (q, t) in enumerate(pairs):
        if only is not None and i not in only:
            continue
        d, oops, st = oracle_py.edlib_align(q, t)
        assert st == 0
        assert dist[i] == d, f"pair {i} ({len(q)} x {len(t)}) distance"
        assert ops[i] == oops, f"pair {i} ({len(q)} x {len(t)}) path"


@pytest.mark.parametrize("error", [0.0, 0.02, 0.12, 0.4])
def test_block_and_chunk_remainders(error):
    rng = np.random.default_rng(11)
    sizes = [1, 15, 16, 17, 31, 63, 64, 65, 128, 129, 447, 448, 449, 1023, 1024, 1025, 2047]
    check([make_pair(rng, n, error) for n in sizes])


@pytest.mark.parametrize("length", [900, 2500, 5000, 9000, 17000])
def test_groups_of_lanes(length):
    rng = np.random.default_rng(length)
    check([make_pair(rng, length, e) for e in (0.01, 0.12, 0.3)])


@pytest.mark.parametrize("band", [1, 60, 900, 3000, 20000, 100000])
def test_band_guesses(band):
    rng = np.random.default_rng(13)
    check([make_pair(rng, n, 0.15) for n in (40, 700, 1700, 2600, 6000)], band)


def test_unequal_lengths():
    rng = np.random.default_rng(17)
    t = random_seq(rng, 9000)
    q = mutate(rng, t, 0.1)
    check([(q[:3000], t), (q, t[:2500]), (q[2000:8500], t[1000:5000]), (q[:70], t),
           (q, t[:33]), (q[:1], t[:4000]), (q[:8800], t[:9]), (q[:6000] + q[7500:], t)])


def test_few_long_pairs_take_a_team():
    rng = np.random.default_rng(19)
    pairs = [make_pair(rng, n, e) for n, e in ((12000, 0.12), (21000, 0.05), (30000, 0.2), (300, 0.1))]
    t = random_seq(rng, 14000)
    pairs.append((mutate(rng, t[:5000] + t[9000:], 0.1), t))
    pairs.append((random_seq(rng, 5000), random_seq(rng, 11000)))
    check(pairs, launches=2)


def test_strips_of_a_team():
    """Bands of more than 16,400 diagonals, too wide for the 256 lanes of half
    a team: strips, dealt to the team's waves."""
    rng = np.random.default_rng(43)
    pairs = [make_pair(rng, 20000, 0.1), make_pair(rng, 17000, 0.3), make_pair(rng, 300, 0.1)]
    t = random_seq(rng, 22000)
    pairs += [(mutate(rng, t[3000:20500], 0.1), t), (t, mutate(rng, t[:18000], 0.1))]
    check(pairs, band=20000, launches=2)


def test_long_pairs_on_one_wave():
    """Pairs that a batch would give to teams, through the entry point that
    runs one wave per pair: strips at the top of the recursion."""
    rng = np.random.default_rng(47)
    pairs = [make_pair(rng, 24000, 0.15), make_pair(rng, 12000, 0.12), make_pair(rng, 19500, 0.05),
             (random_seq(rng, 6000), random_seq(rng, 12000)), make_pair(rng, 300, 0.1)]
    hip = Hip()
    try:
        ops, dist, status = noalloc_align(pairs, hip)
    finally:
        hip.free()
    assert status == [0] * len(pairs)
    compare(pairs, ops, dist)


def test_long_pairs_beside_many_short_ones():
    rng = np.random.default_rng(23)
    pairs = [make_pair(rng, 200, 0.1) for _ in range(2100)]
    pairs[7] = make_pair(rng, 24000, 0.15)
    pairs[900] = (random_seq(rng, 6000), random_seq(rng, 12000))
    check(pairs, only=(0, 7, 8, 900, 2099), launches=2)


@pytest.mark.parametrize("letter", [b"N", b"n", b"R"])
def test_other_bytes_at_chunk_edges(letter):
    rng = np.random.default_rng(29)
    pairs = []
    for n in (40, 1000, 4000):
        t = bytearray(random_seq(rng, n))
        q = bytearray(mutate(rng, bytes(t), 0.1))
        for at in (0, 15, 16, 31, n // 2, n - 1):
            t[at] = letter[0]
        for at in (0, len(q) // 2, len(q) - 1):
            q[at] = letter[0]
        pairs.append((bytes(q), bytes(t)))
    check(pairs)


@pytest.mark.parametrize("length", [63, 64, 65, 129, 500, 1500])
def test_long_gaps(length):
    """Leaves whose paths are mostly gaps: bands of insertions over block
    edges, bands of deletions, and both at the ends of a pair, one wave per
    pair and in teams."""
    rng = np.random.default_rng(length)
    t = random_seq(rng, 8000)
    q = mutate(rng, t, 0.1)
    long_t = random_seq(rng, 14000)
    check([(q[:length], t), (q[-length:], t), (q, t[:length]), (q, t[-length:]),
           (q, t[:4000] + t[4000 + length:]), (q[:4000] + q[4000 + length:], t),
           (random_seq(rng, length), t), (t, random_seq(rng, length)),
           (long_t, random_seq(rng, length)), (random_seq(rng, length), long_t)])


def test_long_gaps_cost_no_more_than_matches():
    """An op of a gap is no round trip of its own: a pair of unequal lengths
    takes less than the square pair of the longer one (up to 2.9 times as long
    with a round trip per op)."""
    rng = np.random.default_rng(31)
    pairs = [make_pair(rng, 8000, 0.12) for _ in range(20)]

    def kernel_ms(batch):
        b = _lib.AlignBatch()
        b.upload(batch)
        times = []
        for _ in range(4):
            b.run()
            times.append(b.stats().kernel_ms)
        b.close()
        return min(times)

    square = kernel_ms(pairs)
    assert kernel_ms([(q, t[:200]) for q, t in pairs]) < square
    assert kernel_ms([(q[:200], t) for q, t in pairs]) < 2 * square
