"""The packed kernel for any penalties (one or two gap pieces) where its tiling
and its rings can go wrong: rings of one slot and of many, shallower and deeper
than the six scores between exchanges; windows that put diagonal 0 or the end
at an edge of its chunks (116 own diagonals); an opening of 0, which it leaves
to the ring kernel.  Scores are whole numbers and must equal the oracle's;
which capacity a pair fits must not depend on the kernel: the range a ring
kernel holds grows by one diagonal per extension after the opening."""
import math
import random

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PENS = [(1, 1, 1), (2, 3, 1), (5, 6, 2), (4, 2, 7), (7, 11, 3), (12, 1, 1), (1, 14, 1), (10, 3, 9), (3, 0, 1), (20, 40, 15),
        (4, 6, 2, 24, 1), (4, 6, 2, 12, 2), (5, 1, 3, 10, 1), (4, 5, 3, 20, 2), (2, 1, 9, 8, 4), (9, 3, 1, 1, 7), (3, 0, 2, 9, 1), (4, 4, 8, 40, 3)]


def say(msg):
    print(f"\n[gpu] {msg}", flush=True)


def seq(rng, n):
    return "".join(rng.choice("ACGT") for _ in range(n))


def edited(rng, s, k):
    s = list(s)
    for _ in range(k):
        i = rng.randrange(len(s))
        c = rng.random()
        if c < 0.34:
            s[i] = rng.choice("ACGT")
        elif c < 0.67:
            s.insert(i, rng.choice("ACGT"))
        elif len(s) > 1:
            del s[i]
    return "".join(s)


def make_pairs(rng):
    pairs = [(p, edited(rng, p, rng.randrange(1 + n // 8))) for n in (1, 15, 16, 17, 33, 128, 300, 700) for p in (seq(rng, n) for _ in range(12))]
    for g in (57, 58, 59, 115, 116, 117, 231, 232):
        p = seq(rng, 200)
        i = rng.randrange(200)
        t = edited(rng, p[:i] + seq(rng, g) + p[i:], 3)
        pairs += [(p, t), (t, p)]
    pairs += [("", ""), ("A", ""), ("", "ACGT" * 10), ("A" * 300, "A" * 290), ("AC" * 200, "CA" * 200), (seq(rng, 150), seq(rng, 500))]
    return pairs


@pytest.mark.parametrize("pen", PENS)
def test_scores_equal_the_oracle(tsu, oracle, pen):
    rng = random.Random(sum(pen))
    pairs = make_pairs(rng)
    two = len(pen) == 5
    want = (oracle.wfa2p_batch if two else oracle.wfa_batch)(pairs, *pen)[0]
    a = tsu.Aligner(*pen[:3], gap_opening2=pen[3], gap_extension2=pen[4]) if two else tsu.Aligner(*pen)
    try:
        b = a.batch(pairs)
        g = math.gcd(*pen)
        fits = None
        for wf in (40, 116, 117, 232, 233, 348, 464, 700, 1100, 2100):
            say(f"{pen} plain wf_length={wf}")
            got = np.empty(len(pairs), np.int32)
            try:
                a.align_plain(b, wf, out=got)
            except tsu.TsuError as err:
                if two and err.status == tsu.TSU_EINVAL:
                    continue   # two pieces: rings wider than LDS are refused as a call
                assert err.status == tsu.TSU_EKOVERFLOW
            ok = got >= 0
            assert (got[~ok] == tsu.TSU_EKOVERFLOW).all()
            assert (got[ok] == want[ok]).all(), np.nonzero(ok & (got != want))[0][:5]
            # a pair whose range stays within the window is never refused
            s = want // g
            half = (s - pen[1] // g) // (pen[2] // g) + 1
            if two:
                half = np.maximum(half, (s - pen[3] // g) // (pen[4] // g) + 1)
            assert ok[half < wf // 2].all()
            fits = ok if fits is None else fits
            assert ok[fits].all()   # a wider window takes what a narrower one does
            fits = ok
        say(f"{pen} batched")
        got, _ = a.align_batched(b)
        assert (got == want).all(), np.nonzero(got != want)[0][:5]
    finally:
        a.close()


@pytest.mark.parametrize("pen", [(5, 6, 2), (4, 5, 3, 20, 2)])
@pytest.mark.parametrize("length,edits", [(9000, 20), (16001, 30), (31990, 40)])
def test_long_accurate_reads(tsu, oracle, pen, length, edits):
    """Packed sequences in LDS, up to the longest it takes; a few pairs and
    (with copies) more than there are CUs, which take fewer waves each."""
    rng = random.Random(length)
    pairs = [(p, edited(rng, p, edits)) for p in (seq(rng, length) for _ in range(3))]
    p = seq(rng, 700) * (length // 700)
    pairs.append((p, edited(rng, p, edits // 2)))
    two = len(pen) == 5
    want = (oracle.wfa2p_batch if two else oracle.wfa_batch)(pairs, *pen)[0]
    a = tsu.Aligner(*pen[:3], gap_opening2=pen[3], gap_extension2=pen[4]) if two else tsu.Aligner(*pen)
    try:
        say(f"{pen} {length} bp, 4 pairs")
        got, _ = a.align_batched(a.batch(pairs))
        assert (got == want).all()
        say("400 pairs")
        got, _ = a.align_plain(a.batch(pairs * 100), 700)
        assert (got == np.tile(want, 100)).all()
    finally:
        a.close()
