"""The blocking of the packed kernel, restated in numpy: chunks of diagonals
that overlap by six at each end, advanced six scores on their own (from
whatever stands beyond their ends) and then given their neighbours' cells
again, with the gap sources kept as max(M[s-3], I[s]) and max(M[s-3], D[s]).
Scores must equal the oracle's."""
import random

import numpy as np
import pytest

NONE = -(1 << 20)
STEP, OWN = 6, 10          # a small chunk shows the same edges
WIDTH = OWN + 2 * STEP


def blocked_score(p, t, beyond):
    P, T = len(p), len(t)
    chunks = (P + T + 1 + OWN - 1) // OWN
    k0 = -P - STEP
    k = k0 + OWN * np.arange(chunks)[:, None] + np.arange(WIDTH)[None, :]
    lim = np.maximum(np.minimum(k + P, T), np.maximum(k, 0))

    def extend(M):
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
    if (M[0][k == T - P] >= T).any():
        return 0
    s = 0
    own = slice(STEP, STEP + OWN)
    while True:
        for _ in range(STEP):
            s += 1
            up = np.concatenate([np.full((chunks, 1), beyond), mi[:, :-1]], axis=1)
            down = np.concatenate([md[:, 1:], np.full((chunks, 1), beyond)], axis=1)
            I, D, X = up + 1, down, M[(s - 2) % 3] + 1
            I, D = np.where(I > lim, NONE, I), np.where(D > lim, NONE, D)
            new = np.maximum(np.maximum(D, X), I)
            new = np.where(new > lim, NONE, new)
            old = M[s % 3]
            mi, md = np.maximum(old, I), np.maximum(old, D)
            M[s % 3] = extend(new)
            at = (T - P) - k0 - STEP
            if M[s % 3][at // OWN, STEP + at % OWN] >= T:
                return s
        for a in (*M, mi, md):
            o = a[:, own].copy()
            a[0, :STEP], a[-1, STEP + OWN:] = NONE, NONE
            a[1:, :STEP] = o[:-1, -STEP:]
            a[:-1, STEP + OWN:] = o[1:, :STEP]


@pytest.mark.parametrize("beyond", [NONE, 0])
def test_blocked_wavefronts_equal_the_oracle(oracle, beyond):
    rng = random.Random(3)
    pairs = [("", ""), ("A", ""), ("", "ACGTACGTACGT"), ("ACGT" * 8, "ACGT" * 8), ("A" * 30, "T" * 30)]
    for _ in range(60):
        p = "".join(rng.choice("ACGT") for _ in range(rng.randint(0, 40)))
        t = list(p)
        for _ in range(rng.randint(0, 8)):
            i = rng.randint(0, len(t))
            t[i:i + rng.randint(0, 6)] = [rng.choice("ACGT") for _ in range(rng.randint(0, 12))]
        pairs.append((p, "".join(t)))
    want, _, _ = oracle.wfa_batch(pairs, 4, 6, 2)
    for (p, t), w in zip(pairs, want):
        assert 2 * blocked_score(p, t, beyond) == w, (p, t)
