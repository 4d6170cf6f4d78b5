"""The packed DP rows at the edges of their forms, against the CPU oracle:
layer lengths around 64 W columns for every strip width W (and past the last
one, where the tiled rows take over), scores whose range just fits or just
exceeds 16 bits, layers with letters other than A, C, G and T, rings of
2 to 16 LDS rows (rows that find no slot go through global memory), and
windows with several predecessors per node.
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


def window(rng, length, depth, error=0.12, exact=()):
    """A window of `length` bases; the layers named in `exact` are cut or
    padded to that many bases."""
    backbone = random_seq(rng, length)
    truth = mutate(rng, backbone, 0.03)
    layers = []
    for k in range(depth):
        begin, end = 0, length - 1
        if k % 5 == 4:
            begin, end = length // 5, length - 1 - length // 7
        seq = mutate(rng, truth[begin:end + 1], error)
        if k < len(exact):
            begin, end = 0, length - 1
            seq = (mutate(rng, truth, error) + random_seq(rng, exact[k]))[:exact[k]]
        layers.append(Layer(seq, random_quality(rng, len(seq)), begin, end))
    return Window(backbone, b"!" * length, layers)


def check(windows, scores=(3, -5, -4), ring=0):
    b = _lib.PoaBatch(*scores, trim=True)
    if ring:
        b.set_tuning(0, 0, ring)
    b.upload(windows)
    b.run(_lib.RH_POA_BATCHED)
    out, status = b.download()
    b.close()
    for i, w in enumerate(windows):
        cons, ost, _, _ = oracle_py.window_consensus(*oracle_args(w), True, *scores)
        assert status[i] == ost, f"window {i} status"
        assert out[i] == cons, f"window {i} consensus"


@pytest.mark.parametrize("columns", [1, 4, 256, 512, 768, 1024, 1280])
def test_layer_lengths_around_a_strip_edge(columns):
    rng = np.random.default_rng(columns)
    exact = [max(1, columns + d) for d in (-2, -1, 0, 1, 2)]
    check([window(rng, max(30, columns), 8, exact=exact) for _ in range(2)])


@pytest.mark.parametrize("scores", [(1, -1, -1), (5, -4, -8), (30, -20, -25), (127, -127, -20),
                                    (1, -128, -128), (3, -5, 0)])
def test_score_ranges_around_16_bits(scores):
    rng = np.random.default_rng(17)
    check([window(rng, n, 10) for n in (40, 250, 480, 700)], scores)


@pytest.mark.parametrize("ring", [2, 3, 5, 16])
def test_rows_without_an_lds_slot(ring):
    rng = np.random.default_rng(23)
    check([window(rng, n, 24, error=0.2) for n in (120, 505, 900)], ring=ring)


def test_letters_other_than_acgt():
    rng = np.random.default_rng(29)
    wins = [window(rng, 300, 12) for _ in range(4)]
    for w in wins[:3]:
        for k in (1, 4, 7):
            seq = bytearray(w.layers[k].sequence)
            for at in rng.integers(0, len(seq), size=5):
                seq[at] = ord("N")
            w.layers[k].sequence = bytes(seq)
    backbone = bytearray(wins[3].backbone)
    backbone[10:14] = b"NNNN"
    wins[3].backbone = bytes(backbone)
    check(wins)


@pytest.mark.parametrize("length", [60, 300, 600, 900, 1150])
def test_odd_letters_at_every_strip_width(length):
    """Layers with other letters, some at the strip edges, some equal to the
    backbone's, beside plain layers of the same window."""
    rng = np.random.default_rng(length)
    win = window(rng, length, 6)
    backbone = bytearray(win.backbone)
    backbone[length // 2] = ord("N")
    win.backbone = bytes(backbone)
    for k in (0, 2, 3):
        seq = bytearray(win.layers[k].sequence)
        for at in [0, len(seq) - 1, len(seq) // 2, *rng.integers(0, len(seq), size=6)]:
            seq[at] = ord("N") if at % 3 else ord("a")
        win.layers[k].sequence = bytes(seq)
    check([win])


def test_many_predecessors():
    """Long random deletions give nodes with far more than four in-edges."""
    rng = np.random.default_rng(31)
    wins = []
    for _ in range(3):
        backbone = random_seq(rng, 400)
        layers = []
        for k in range(40):
            cut = int(rng.integers(0, 150))
            seq = mutate(rng, backbone[:200 - cut] + backbone[200:], 0.03)
            layers.append(Layer(seq, None, 0, 399))
        wins.append(Window(backbone, b"!" * 400, layers))
    check(wins)


def run_phases(windows, ring=0):
    b = _lib.PoaBatch(3, -5, -4, trim=True)
    if ring:
        b.set_tuning(0, 0, ring)
    for _ in range(2):  # (the first run also loads the code)
        b.upload(windows)
        b.run(_lib.RH_POA_BATCHED)
    phases = b.phase_seconds()
    b.close()
    return phases


def lower(w):
    layers = [Layer(l.sequence.lower(), l.quality, l.begin, l.end) for l in w.layers]
    return Window(w.backbone.lower(), w.backbone_quality, layers)


@pytest.mark.parametrize("form", ["global rows", "lower case"])
def test_rows_of_the_general_form_trace_in_tiles(form):
    """The moves of rows in global memory and of rows with another letter are
    as cheap to follow as the others' (one round trip per move took 5 and 8
    times as long; the bound leaves room for a busy device)."""
    rng = np.random.default_rng(37)
    wins = [window(rng, 500, 12) for _ in range(24)] * 50
    plain = run_phases(wins)["traceback"]
    if form == "global rows":
        general = run_phases(wins, ring=2)["traceback"]
    else:
        general = run_phases([lower(w) for w in wins])["traceback"]
    assert general < 2 * plain


def test_rows_of_another_letter_stay_near_the_others():
    """The DP of rows of other letters costs about what the others' does (the
    general form took 3.3 times as long, a row of byte compares 2.4)."""
    rng = np.random.default_rng(41)
    wins = [window(rng, 500, 12) for _ in range(24)] * 50
    assert run_phases([lower(w) for w in wins])["dp"] < 2.4 * run_phases(wins)["dp"]


@pytest.mark.parametrize("length", [60, 300, 600, 900, 1150])
@pytest.mark.parametrize("ring", [0, 2])
def test_windows_of_two_cases(length, ring):
    """Rows of other letters beside the rest, with and without an LDS slot:
    layers in lower case, half in lower case, and in upper case."""
    rng = np.random.default_rng(length + 1)
    win = window(rng, length, 9, error=0.2)
    half = length // 2
    win.backbone = win.backbone[:half].lower() + win.backbone[half:]
    for k, layer in enumerate(win.layers):
        seq = layer.sequence
        layer.sequence = (seq.lower(), seq[:half].lower() + seq[half:], seq)[k % 3]
    check([win, lower(win)], ring=ring)
