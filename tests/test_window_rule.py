"""The packed kernel's rule for pairs that leave their capacity against the
ring kernels' ranges, for every capacity of small pairs."""
import random

import pytest

from window_model import first_pass, passes, run


def pairs(rng, n, longest):
    out = [("A" * 9, "A" * 9), ("A", "ACGTACGT"), ("ACGTACGTAC", "C"), ("", "ACG"), ("ACG", "")]
    for _ in range(n):
        p = "".join(rng.choice("ACGT") for _ in range(rng.randint(1, longest)))
        if rng.random() < 0.3:
            p = (p[:3] * longest)[:len(p)]
        t = list(p)
        for _ in range(rng.randint(0, 5)):
            i = rng.randint(0, len(t))
            t[i:i + rng.randint(0, 8)] = [rng.choice("ACGT") for _ in range(rng.randint(0, 9))]
        out.append((p, "".join(t)))
    return out


@pytest.mark.parametrize("x,pieces", [
    (5, [(6, 2)]), (4, [(5, 3)]), (1, [(1, 1)]), (7, [(9, 2)]), (2, [(1, 5)]),
    (2, [(3, 1), (12, 1)]), (4, [(6, 2), (24, 1)]), (3, [(2, 3), (9, 2)]), (2, [(1, 1), (3, 4)]), (5, [(1, 2), (4, 7)]),
])
def test_edge_cells_tell_when_the_range_leaves(oracle, x, pieces):
    rng = random.Random(x + 10 * len(pieces))
    both = [0, 0]
    for p, t in pairs(rng, 60, 28):
        score, ranges, cells = run(p, t, pieces, x)
        if len(pieces) == 1:
            assert score == oracle.wfa_batch([(p, t)], x, *pieces[0])[0][0], (p, t)
        for W in range(1, len(p) + len(t) + 4):
            over = passes(p, t, W, ranges)
            assert over == (first_pass(p, t, W, pieces, cells) <= score), (p, t, W)
            both[over] += 1
    assert min(both) > 100
