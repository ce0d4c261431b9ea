"""The packed kernel (4/6/2; two diagonals per lane and register) at the sizes
where its tiling can go wrong: end diagonals at the edges of chunks (116 own
diagonals, 6 copies at each end) and of lanes, sequence lengths around its
16-base words, every window and wave count, sequences expanded in LDS (short
ones) and packed (long ones in narrow windows), plain, queue-fed and with backtrace records.  Scores
and CIGARs are whole numbers and must equal the oracle's."""
import random

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


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
        else:
            del s[i]
    return "".join(s)


def check(aligner, oracle, pairs, wf_length):
    want, ops, _ = oracle.wfa_batch(pairs, 4, 6, 2, cigar=True)
    b = aligner.batch(pairs)
    say(f"plain wf_length={wf_length}, {len(pairs)} pairs")
    got, _ = aligner.align_plain(b, wf_length)
    assert (got == want).all(), np.nonzero(got != want)[0][:5]
    say("batched")
    got, _ = aligner.align_batched(b)
    assert (got == want).all(), np.nonzero(got != want)[0][:5]
    say("CIGARs")
    got, cig, _ = aligner.align_cigar(b)
    assert (got == want).all(), np.nonzero(got != want)[0][:5]
    bad = [i for i in range(len(pairs)) if cig[i] != oracle.rle(ops[i])]
    assert not bad, bad[:5]


@pytest.mark.parametrize("wf_length,base,gaps", [
    (64, 40, (0, 1, 5, 14)),
    (128, 100, (0, 1, 30, 50)),
    (256, 150, (57, 58, 59, 63, 64, 65, 90)),
    (512, 300, (57, 58, 115, 116, 117, 121, 122, 173, 174, 175, 200)),
    (1024, 500, (57, 58, 173, 174, 231, 232, 233, 347, 348, 400)),
    (2000, 1500, (115, 116, 231, 232, 700)),
    (4096, 2500, (115, 116, 117, 463, 464, 465, 1200)),
    (8192, 3500, (927, 928, 929, 2500)),
    (16384, 4500, (1855, 1856, 1857, 3500)),
])
def test_end_diagonal_at_chunk_edges(aligner, oracle, wf_length, base, gaps):
    """One long gap (either way) puts the end diagonal at a chosen place."""
    rng = random.Random(wf_length)
    pairs = []
    for g in gaps:
        for _ in range(2):
            p = seq(rng, base)
            i = rng.randrange(base)
            t = edited(rng, p[:i] + seq(rng, g) + p[i:], 3)
            pairs += [(p, t), (t, p)]
    check(aligner, oracle, pairs, wf_length)


@pytest.mark.parametrize("length", [1, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 255, 257, 1000])
def test_lengths_around_words(aligner, oracle, length):
    rng = random.Random(length)
    pairs = [(p, edited(rng, p, 1 + length // 12) or "A") for p in (seq(rng, length) for _ in range(24))]
    pairs += [(seq(rng, length), seq(rng, rng.randint(1, length))) for _ in range(8)]
    pairs += [("A" * length, "A" * max(1, length - 3)), ("AC" * length, "CA" * length), ("A" * length, "T" * length)]
    check(aligner, oracle, pairs, 2 * length + 400)


@pytest.mark.parametrize("length,edits,wf_length", [(6000, 12, 128), (9000, 30, 512), (16001, 40, 512), (31990, 60, 1024),
                                                    (31990, 300, 4096)])
def test_long_accurate_reads(aligner, oracle, length, edits, wf_length):
    """Long runs (extended by the whole wave) on packed sequences, up to the
    longest the kernel takes."""
    rng = random.Random(length + edits)
    pairs = [(p, edited(rng, p, edits)) for p in (seq(rng, length) for _ in range(4))]
    p = seq(rng, 700) * (length // 700)          # repeats: many cells extend at once
    pairs.append((p, edited(rng, p, edits // 2)))
    check(aligner, oracle, pairs, wf_length)


def test_extensions_longer_than_a_record_holds(aligner, oracle):
    """Runs of 4,094 to 12,000 matches: a record holds lengths below 4,095,
    the others are in the list behind the records."""
    rng = random.Random(8)
    pairs = []
    for n in (4093, 4094, 4095, 4096, 4097, 8191, 12000):
        p, q = seq(rng, n), seq(rng, 300)
        pairs += [(q + "A" + p + "C" + q, q + "T" + p + "G" + q), (p + q, p + "ACGTAC" + q), ("A" * n + q, "A" * (n + 3) + q)]
    check(aligner, oracle, pairs, 512)


@pytest.mark.parametrize("pairs_n,window", [(300, 512), (300, 1024), (200, 2048), (100, 4096), (40, 8192), (2, 24576)])
def test_waves_per_pair_follow_the_pair_count(aligner, oracle, pairs_n, window):
    """Few pairs take more waves each (5 or 3 chunks a wave instead of 9), and
    pairs wider than 16,384 diagonals the widest window: the same scores."""
    rng = random.Random(window)
    bound = {512: 512, 1024: 1024, 2048: 2048, 4096: 4096, 8192: 8192, 24576: 16383}[window]
    if window == 24576:
        pairs = [(seq(rng, 12_500), seq(rng, 12_000)) for _ in range(pairs_n)]
    else:
        base = [seq(rng, bound - 60) for _ in range(20)]
        pairs = [(p, edited(rng, p, rng.randrange(1, window // 16))) for p in (rng.choice(base) for _ in range(pairs_n))]
        pairs = [(p, t) for p, t in pairs if max(len(p), len(t)) <= bound]
    want, _, _ = oracle.wfa_batch(pairs, 4, 6, 2)
    aligner.set_tune_table([{"waves_per_pair": 1, "capacity": window, "bucket_bound": bound}])
    try:
        b = aligner.batch(pairs)
        say(f"{len(pairs)} pairs in {window} diagonals, batched")
        got, _ = aligner.align_batched(b)
        assert (got == want).all(), np.nonzero(got != want)[0][:5]
        say("the first eight")
        got, _ = aligner.align_batched(aligner.batch(pairs[:8]))
        assert (got == want[:8]).all()
    finally:
        aligner.set_tune_table([])
