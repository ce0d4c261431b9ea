"""CIGAR calls most of whose pairs overflow their first window: recorded again
in twice as many diagonals, all at once where their state allows, and never
left to a score pass for want of run words."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"\n[gpu] {msg}", flush=True)


def unrelated(rng, n, length):
    a = ["".join(x) for x in rng.choice(list("ACGT"), (2 * n, length))]
    return list(zip(a[:n], a[n:]))


def check(aligner, oracle, pairs):
    want, ops, _ = oracle.wfa_batch(pairs, 4, 6, 2, cigar=True)
    got, cig, t = aligner.align_cigar(aligner.batch(pairs))
    assert (got == want).all(), np.nonzero(got != want)[0][:5]
    bad = [i for i in range(len(pairs)) if cig[i] != oracle.rle(ops[i])]
    assert not bad, bad[:5]
    return t


@pytest.mark.parametrize("n,length", [(3000, 120), (3000, 250), (1500, 500)])
def test_unrelated_pairs_take_two_record_launches(aligner, oracle, n, length):
    pairs = unrelated(np.random.default_rng(length), n, length)
    say(f"CIGARs of {n} unrelated pairs of {length} bp")
    t = check(aligner, oracle, pairs)
    assert t["record_launches"] == 2 and t["launches"] == 2, t


@pytest.mark.parametrize("budget_mib", [0, 256, 40])
def test_unrelated_pairs_beside_ordinary_ones(tsu, oracle, budget_mib):
    """Several length buckets, the unrelated pairs in some of them, with the
    state of all launches at once and with a few at a time."""
    rng = np.random.default_rng(9)
    pairs = []
    for length, n, kind in ((100, 800, "u"), (400, 400, "o"), (500, 300, "u"), (900, 200, "u"), (3000, 60, "o"), (3000, 12, "u")):
        if kind == "u":
            pairs += unrelated(rng, n, length)
        else:
            pairs += tsu.Dataset.generate(n, seed=length, len_min=length, err_min=0.05).pairs()
    a = tsu.Aligner(4, 6, 2)
    try:
        a.set_cigar_memory(a.CIGAR_AUTO, 0, budget_mib << 20)
        for again in range(2):
            say(f"CIGARs of {len(pairs)} pairs, budget {budget_mib} MiB, call {again}")
            t = check(a, oracle, pairs)
            if budget_mib:
                assert t["state_bytes"] <= budget_mib << 20
    finally:
        a.close()
