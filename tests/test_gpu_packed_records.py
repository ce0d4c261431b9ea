"""CIGARs of the packed kernel (4/6/2) where its 16-bit records do not hold an
extension's length (4,095 bases and more): such lengths are in a list keyed by
score and diagonal.  CIGARs are compared with the oracle's."""
import random

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"\n[gpu] {msg}", flush=True)


def seq(rng, n):
    return "".join(rng.choice("ACGT") for _ in range(n))


def other(rng, c):
    return rng.choice([x for x in "ACGT" if x != c])


def substituted(rng, s, *places):
    for i in places:
        s = s[:i] + other(rng, s[i]) + s[i + 1:]
    return s


def gap_or_mismatch_first(rng, gap, same, tail):
    """A gap of `gap` bases and a mismatch in either order, the same cost: on
    the end diagonal the gap's cell lies `same` bases further than the
    mismatch's, and both run into one match of `tail` bases."""
    head, a, w, end = seq(rng, 900), rng.choice("ACGT"), seq(rng, same), seq(rng, tail)
    p = substituted(rng, head, 300, 600) + other(rng, a) + w + seq(rng, gap - same - 1) + other(rng, a) + w + end
    return p, head + a + w + end


def gap_at_repeat(rng, gap, tail):
    """The same with a substitution before the gap's other end."""
    t = seq(rng, 100 + tail)
    p = (t[:100] + other(rng, t[100]) + t[101:110] + other(rng, t[110]) + seq(rng, gap - 11) + other(rng, t[100]) + t[101:])
    return substituted(rng, p, 20, 60), t


def check_cigars(aligner, oracle, pairs, entries=()):
    want, ops, _ = oracle.wfa_batch(pairs, 4, 6, 2, cigar=True)
    aligner.set_tune_table(list(entries))
    try:
        got, cig, t = aligner.align_cigar(aligner.batch(pairs))
    finally:
        aligner.set_tune_table([])
    assert (got == want).all(), np.nonzero(got != want)[0][:5]
    bad = [i for i in range(len(pairs)) if cig[i] != oracle.rle(ops[i])]
    assert not bad, (len(bad), bad[:5], cig[bad[0]], oracle.rle(ops[bad[0]]))
    return t


@pytest.mark.parametrize("window", [128, 256, 512, 1024, 2048, 4096, 8192])
def test_long_extensions_at_chunk_edges(aligner, oracle, window):
    """End diagonals in and beside every copy of a neighbour's diagonals at the
    first chunk edges on both sides of diagonal 0, in one wave and several."""
    rng = random.Random(window)
    pairs = []
    for gap in [g for g in [*range(30, 70), *range(160, 180)] if g < window // 2 - 8]:
        for p, t in (gap_or_mismatch_first(rng, gap, 4, 4596), gap_or_mismatch_first(rng, gap, 1 + gap % 6, 4200),
                     gap_at_repeat(rng, gap, 5900)):
            pairs += [(p, t), (t, p)]
    say(f"CIGARs of {len(pairs)} pairs in {window} diagonals")
    check_cigars(aligner, oracle, pairs, [{"waves_per_pair": 1, "capacity": window, "bucket_bound": 8192}])


@pytest.mark.parametrize("edits", [40, 100])
def test_window_widened_by_another_pair(aligner, oracle, edits):
    """The pairs' own scores fit 128 diagonals, but a pair with more edits in
    the call takes all to a window of several chunks."""
    rng = random.Random(edits)
    pairs = []
    for gap in (50, 52, 53, 54):
        for p, t in (gap_or_mismatch_first(rng, gap, 4, 4596), gap_at_repeat(rng, gap, 5900)):
            pairs += [(p, t), (t, p)]
    wide = seq(rng, 5000)
    pairs.append((wide, substituted(rng, wide, *rng.sample(range(5000), edits))))
    say(f"CIGARs of {len(pairs)} pairs, one with {edits} substitutions")
    check_cigars(aligner, oracle, pairs)


def low_complexity(rng):
    """Tracts of short periods, where cells of many diagonals extend by 4,095
    bases and more."""
    h, pairs = seq(rng, 10), []
    for unit in (1, 5):
        u, d, end = seq(rng, unit), [seq(rng, 100) for _ in range(4)], seq(rng, 4800)
        tract = (u * 5000)[:5000]
        pairs.append((d[0] + tract + d[1] + end, d[2] + tract + d[3] + end))
    segments = ("A" * 4600 + "C") * 3
    pairs.append((h + "C" + segments + h, h + "G" + "A" * 400 + segments + h))
    pairs.append((h + "C" + "ACAC" * 3900, h + "G" + "ACAC" * 3960))
    return pairs


@pytest.mark.parametrize("window", [0, 1024, 4096, 8192, 16384])
def test_many_long_extensions(aligner, oracle, window):
    """Hundreds to thousands of listed extensions, the walk's own among the
    last, beside ordinary pairs; windows by the library (0) and pinned."""
    rng = random.Random(31)
    pairs = [q for p, t in low_complexity(rng) for q in ((p, t), (t, p))]
    for n in (900, 5000, 9000):
        p = seq(rng, n)
        pairs.append((p, substituted(rng, p, *rng.sample(range(n), n // 40))))
    say(f"CIGARs of {len(pairs)} pairs, window {window}")
    check_cigars(aligner, oracle, pairs,
                 [{"waves_per_pair": 1, "capacity": window, "bucket_bound": b} for b in (8192, 16383)] if window else [])


def test_more_long_extensions_than_the_list_holds(aligner, oracle):
    """Three segments of a homopolymer and a gap of 500 in 1,024 diagonals: 2,409
    listed extensions where one wave's 9 chunks have room for 2,304 (over 512
    pairs, so a pair has one wave), and the walk needs the last.  Such a pair
    is recorded with offsets; the call's other pairs stay where they were."""
    rng = random.Random(47)
    h, segments = seq(rng, 10), ("A" * 4900 + "C") * 3
    pair = (h + "C" + segments + h, h + "G" + "A" * 500 + segments + h)
    pairs = [pair, pair[::-1]]
    for _ in range(520):
        p = seq(rng, rng.randint(8200, 8300))
        pairs.append((p, substituted(rng, p, *rng.sample(range(8000), 3))))
    say(f"CIGARs of {len(pairs)} pairs in 1,024 diagonals")
    t = check_cigars(aligner, oracle, pairs, [{"waves_per_pair": 1, "capacity": 1024, "bucket_bound": 16383}])
    assert t["kernels"] == {"reg1", "lds"}
    say("with checkpoints where records do not fit")
    aligner.set_cigar_memory(aligner.CIGAR_AUTO, 0, 8 << 20)
    try:
        t = check_cigars(aligner, oracle, pairs[:2], [{"waves_per_pair": 1, "capacity": 1024, "bucket_bound": 16383}])
    finally:
        aligner.set_cigar_memory()
    assert t["state_bytes"] <= 8 << 20


def test_scored_pairs_of_the_widest_window(aligner, oracle):
    """Unrelated pairs of 7,000 bases (8,193 to 16,384 diagonals), scored first
    since their bucket is tuned to the LDS kernel: recorded by the packed
    kernel's widest window."""
    rng = random.Random(7)
    pairs = [(seq(rng, 7000), seq(rng, 7000 - 40 * i)) for i in range(3)]
    say("CIGARs of 3 unrelated pairs, scored first")
    t = check_cigars(aligner, oracle, pairs, [{"waves_per_pair": 4, "capacity": 0, "bucket_bound": 8192}])
    assert t["kernels"] == {"ml16"}, t["kernels"]
