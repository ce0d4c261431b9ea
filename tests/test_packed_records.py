"""Backtrace records of the packed kernel, restated in numpy with small chunks
and short lengths: a cell's gap bits where the gap comes from, the lengths of
extensions in the records, and those a record does not hold in a list keyed by
score and diagonal.  The walk over them must give the oracle's CIGAR.

A chunk's copies of its neighbours' cells are inexact between exchanges, so
only the owner of a diagonal may list an extension."""
import random

import numpy as np
import pytest

NONE = -(1 << 20)
STEP, OWN, LONG = 6, 10, 5   # LONG: the record's mark of a listed length
WIDTH = OWN + 2 * STEP


def record(p, t, beyond, list_copies=False):
    """(score, first own diagonal, records by score, the list in append order)."""
    P, T = len(p), len(t)
    chunks = (P + T + 1 + OWN - 1) // OWN
    k0 = -P
    k = k0 - STEP + OWN * np.arange(chunks)[:, None] + np.arange(WIDTH)[None, :]
    lim = np.maximum(np.minimum(k + P, T), np.maximum(k, 0))
    own = slice(STEP, STEP + OWN)
    recs, listed = {}, []

    def extend(M):
        M = M.copy()
        for c, j in zip(*np.nonzero((M >= 0) & (M < lim))):
            h = M[c, j]
            v = h - k[c, j]
            while h < lim[c, j] and 0 <= v < P and p[v] == t[h]:
                h, v = h + 1, v + 1
            M[c, j] = h
        return M

    M = [np.full(k.shape, NONE) for _ in range(3)]
    mi, md = np.full(k.shape, NONE), np.full(k.shape, NONE)
    M[0][k == 0] = 0
    M[0] = extend(M[0])
    if P == T and M[0][k == 0][0] == T:
        return 0, k0, recs, listed
    s = 0
    while True:
        block = []
        for _ in range(STEP):
            s += 1
            up = np.concatenate([np.full((chunks, 1), beyond), mi[:, :-1]], axis=1)
            down = np.concatenate([md[:, 1:], np.full((chunks, 1), beyond)], axis=1)
            I, D, X = up + 1, down, M[(s - 2) % 3] + 1
            I, D = np.where(I > lim, NONE, I), np.where(D > lim, NONE, D)
            before = np.maximum(np.maximum(D, X), I)
            before = np.where(before > lim, NONE, before)
            old = M[s % 3]
            mi, md = np.maximum(old, I), np.maximum(old, D)
            flags = (before != X) * 1 + (before != D) * 2 + (mi != I) * 4 + (md != D) * 8
            M[s % 3] = extend(before)
            length = M[s % 3] - before
            recs[s] = (np.minimum(length, LONG) * 16 + flags)[:, own].ravel()
            for c, j in zip(*np.nonzero((length >= LONG) & (before >= 0))):
                if list_copies or STEP <= j < STEP + OWN:
                    block.append((c, s, int(k[c, j]), int(length[c, j])))
            at = (T - P) - k0
            if M[s % 3][at // OWN, STEP + at % OWN] >= T:
                # a chunk runs its six scores before the next one starts
                listed += [e[1:] for e in sorted(block, key=lambda e: e[0])]
                return s, k0, recs, listed
        listed += [e[1:] for e in sorted(block, key=lambda e: e[0])]
        for a in (*M, mi, md):
            o = a[:, own].copy()
            a[0, :STEP], a[-1, STEP + OWN:] = NONE, NONE
            a[1:, :STEP] = o[:-1, -STEP:]
            a[:-1, STEP + OWN:] = o[1:, :STEP]


def walk(p, t, score, k0, recs, listed):
    """Operations from the start, as the kernel walks them from the end."""
    k, off, s, kind, ops = len(t) - len(p), len(t), score, 0, []
    while off - k > 0 and off > 0 and s > 0:
        if kind == 0:
            r = int(recs[s][k - k0])
            e = r >> 4
            if e == LONG:
                e = next(n for ss, kk, n in listed if (ss, kk) == (s, k))
            ops += ["M"] * e
            off -= e
            if off - k <= 0 or off <= 0:
                break
            if not r & 1:
                ops.append("X")
                s, off = s - 2, off - 1
                continue
            kind = 1 if r & 2 else 2
        if kind == 1:
            ops.append("I")
            k, off = k - 1, off - 1
        else:
            ops.append("D")
            k += 1
        if int(recs[s - 1][k - k0]) & (4 if kind == 1 else 8):
            s, kind = s - 4, 0
        else:
            s -= 1
    if s == 0:
        n = min(off - k, off)
        ops += ["M"] * n
        off -= n
    ops += ["I"] * off if off - k == 0 else ["D"] * (off - k)
    return "".join(reversed(ops))


def pairs():
    rng = random.Random(5)
    out = [("ACGT" * 8, "ACGT" * 8), ("A" * 30, "A" * 41), ("AC" * 20, "CA" * 17)]
    for _ in range(250):
        unit = "".join(rng.choice("ACGT") for _ in range(rng.choice([1, 2, 3, 30, 60])))
        p = (unit * 60)[:rng.randint(1, 60)]
        t = list(p)
        for _ in range(rng.randint(0, 6)):
            i = rng.randint(0, len(t))
            t[i:i + rng.randint(0, 12)] = [rng.choice("ACGT") for _ in range(rng.randint(0, 14))]
        if t:
            out += [(p, "".join(t)), ("".join(t), p)]
    return out


@pytest.mark.parametrize("beyond", [NONE, 0])
def test_walk_over_records_equals_the_oracle(oracle, beyond):
    cases = pairs()
    want, ops, _ = oracle.wfa_batch(cases, 4, 6, 2, cigar=True)
    copies_wrong = 0
    for (p, t), w, o in zip(cases, want, ops):
        score, k0, recs, listed = record(p, t, beyond)
        assert 2 * score == w, (p, t)
        assert len(set(e[:2] for e in listed)) == len(listed)
        assert walk(p, t, score, k0, recs, listed) == o, (p, t)
        copies_wrong += walk(p, t, *record(p, t, beyond, list_copies=True)) != o
    assert copies_wrong > 0  # the rule is needed: copies that list give other CIGARs
