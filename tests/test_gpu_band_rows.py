"""Band rows at the edges of their form, against the CPU oracle. The layers
have few errors, so that the best path stays well inside 256 columns around
the diagonal and the banded result is the exact one: layer lengths around the
shortest banded one and around whole strips, more columns than the unbanded
packed rows hold, rings so small that rows go through global memory, letters
other than A, C, G and T, and nodes with more than four predecessors.
"""
import sys

import numpy as np
import pytest

from racon_amd import _lib
from racon_amd._lib import Layer, Window
from synth import mutate, oracle_args, random_quality, random_seq

sys.path.insert(0, _lib.PKG_DIR + "/../oracle")
import oracle_py  # noqa: E402

pytestmark = pytest.mark.gpu


def window(rng, length, depth, exact=()):
    backbone = random_seq(rng, length)
    layers = []
    for k in range(depth):
        seq = mutate(rng, backbone, 0.03)
        if k < len(exact):
            seq = (seq + random_seq(rng, 8))[:exact[k]]
        layers.append(Layer(seq, random_quality(rng, len(seq)), 0, length - 1))
    return Window(backbone, b"!" * length, layers)


def check(windows, scores=(3, -5, -4), ring=0):
    b = _lib.PoaBatch(*scores, trim=True)
    b.set_band(256)
    if ring:
        b.set_tuning(0, 0, ring)
    b.upload(windows)
    b.run(_lib.RH_POA_BATCHED)
    out, status = b.download()
    reruns = b.stats().band_reruns
    b.close()
    assert reruns == 0  # (the band rows themselves gave these results)
    for i, w in enumerate(windows):
        cons, ost, _, _ = oracle_py.window_consensus(*oracle_args(w), True, *scores)
        assert status[i] == ost, f"window {i} status"
        assert out[i] == cons, f"window {i} consensus"


@pytest.mark.parametrize("columns", [257, 260, 263, 384, 512, 1024, 1283, 1600])
def test_layer_lengths(columns):
    rng = np.random.default_rng(columns)
    exact = [columns + d for d in (-1, 0, 1, 2, 3)]
    check([window(rng, columns, 8, exact) for _ in range(2)])


@pytest.mark.parametrize("scores", [(1, -1, -1), (5, -4, -8)])
def test_scores(scores):
    rng = np.random.default_rng(5)
    check([window(rng, n, 12) for n in (300, 505, 800)], scores)


@pytest.mark.parametrize("ring", [2, 3, 16])
def test_rows_without_an_lds_slot(ring):
    rng = np.random.default_rng(23)
    check([window(rng, n, 16) for n in (270, 505, 900)], ring=ring)


def test_letters_other_than_acgt():
    rng = np.random.default_rng(29)
    wins = [window(rng, 300, 10) for _ in range(3)]
    for k in (1, 4, 7):
        seq = bytearray(wins[0].layers[k].sequence)
        for at in rng.integers(0, len(seq), size=4):
            seq[at] = ord("N")
        wins[0].layers[k].sequence = bytes(seq)
    backbone = bytearray(wins[1].backbone)
    backbone[10:12] = b"NN"
    wins[1].backbone = bytes(backbone)
    check(wins)


def test_many_predecessors():
    rng = np.random.default_rng(31)
    wins = []
    for _ in range(3):
        backbone = random_seq(rng, 400)
        layers = []
        for _ in range(24):
            cut = int(rng.integers(0, 30))
            seq = mutate(rng, backbone[:200 - cut] + backbone[200:], 0.02)
            layers.append(Layer(seq, None, 0, 399))
        wins.append(Window(backbone, b"!" * 400, layers))
    check(wins)


def consensus(windows, ring):
    b = _lib.PoaBatch(3, -5, -4, trim=True)
    b.set_band(256)
    if ring:
        b.set_tuning(0, 0, ring)
    b.upload(windows)
    b.run(_lib.RH_POA_BATCHED)
    out, _ = b.download()
    b.close()
    return out


@pytest.mark.parametrize("ring", [0, 2])
def test_rows_of_another_letter(ring):
    """Alignments depend on which letters are equal only: windows in lower
    case give the same consensus in lower case, also where the band is an
    approximation (the oracle has no band)."""
    rng = np.random.default_rng(37)
    wins = [window(rng, n, 9) for n in (280, 505, 900, 1400)]
    lower = [Window(w.backbone.lower(), w.backbone_quality,
                    [Layer(l.sequence.lower(), l.quality, l.begin, l.end) for l in w.layers])
             for w in wins]
    assert consensus(lower, ring) == [c.lower() for c in consensus(wins, ring)]
