"""Which pairs fit a capacity of the plain form, for penalties other than 4/6/2
and with two gap pieces: the ring kernels' answer for every capacity (and the
2-piece register kernel's where its window is wider), scores equal to the
oracle's for those that fit.  Expected answers from window_model.py."""
import random

import numpy as np
import pytest

from window_model import passes, run, touches

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"\n[gpu] {msg}", flush=True)


def make(tsu, x, pieces):
    (o, e), rest = pieces[0], pieces[1:]
    return tsu.Aligner(x, o, e, **({"gap_opening2": rest[0][0], "gap_extension2": rest[0][1]} if rest else {}))


def small_pairs(rng, n, longest):
    out = [("A" * 9, "A" * 9), ("A", "ACGTACGT"), ("ACGTACGTAC", "C")]
    for i in range(n):
        size = rng.randint(1, longest if i % 3 else 24)
        p = "".join(rng.choice("ACGT") for _ in range(size))
        if i % 4 == 0:
            p = (p[:3] * longest)[:size]
        t = list(p)
        for _ in range(rng.randint(0, 5)):
            at = rng.randint(0, len(t))
            t[at:at + rng.randint(0, size // 3)] = [rng.choice("ACGT") for _ in range(rng.randint(0, size // 2 + 3))]
        out.append((p, "".join(t) or "A"))
    return out


@pytest.mark.parametrize("x,pieces", [
    (5, [(6, 2)]), (4, [(5, 3)]), (1, [(1, 1)]), (7, [(9, 2)]), (2, [(1, 5)]),
    (2, [(1, 1), (3, 4)]), (3, [(2, 3), (9, 2)]), (5, [(1, 2), (4, 7)]),
])
def test_every_capacity_of_small_pairs(tsu, x, pieces):
    rng = random.Random(100 * x + len(pieces))
    pairs = small_pairs(rng, 42, 100)
    model = [run(p, t, pieces, x) for p, t in pairs]
    a = make(tsu, x, pieces)
    try:
        b = a.batch(pairs)
        say(f"penalties {x} {pieces}, {len(pairs)} pairs, capacities 8 (the least) to 240")
        for W in [*range(8, 64), *range(64, 240, 7), 115, 116, 117, 231, 232, 233]:
            got, _ = a.align_plain(b, W, raise_on_error=False)
            want = [tsu.TSU_EKOVERFLOW if passes(p, t, W, r) else s for (p, t), (s, r, _) in zip(pairs, model)]
            assert list(got) == want, (W, [i for i, (g, w) in enumerate(zip(got, want)) if g != w][:5])
    finally:
        a.close()


@pytest.mark.parametrize("x,pieces,capacities", [
    (4, [(6, 2), (24, 1)], (490, 509, 510, 511, 512, 513)), (2, [(3, 1), (12, 1)], (510, 511, 512)),
    (4, [(6, 3), (24, 1)], (511, 512)), (4, [(6, 2), (24, 1)], (766, 767, 768)),
])
def test_capacities_at_the_register_window(tsu, x, pieces, capacities):
    """A gap to the edge of the window and substitutions before it; 513 to 768
    diagonals take one of 768."""
    rng = random.Random(capacities[-1])
    half = capacities[-1] // 2
    pairs = []
    for gap in (half - 12, half - 3, half - 2, half - 1, half):
        p = "".join(rng.choice("ACGT") for _ in range(half + 60))
        t = p[:10] + ("A" if p[10] != "A" else "C") + p[11:40] + "".join(rng.choice("ACGT") for _ in range(gap)) + p[40:]
        pairs += [(p, t), (t, p)]
    model = [run(p, t, pieces, x) for p, t in pairs]
    a = make(tsu, x, pieces)
    try:
        b = a.batch(pairs)
        signs = set()
        for W in capacities:
            say(f"penalties {x} {pieces}, {len(pairs)} pairs, capacity {W}")
            got, _ = a.align_plain(b, W, raise_on_error=False)
            win = 512 if W <= 512 else 768
            want = [s if not passes(p, t, W, r) or not touches(p, t, win, c) else tsu.TSU_EKOVERFLOW
                    for (p, t), (s, r, c) in zip(pairs, model)]
            assert list(got) == want, (W, [i for i, (g, w) in enumerate(zip(got, want)) if g != w][:5])
            signs |= set(np.sign(want))
        assert len(signs) == 2
    finally:
        a.close()


def test_overflowing_pairs_cost_one_launch(tsu):
    """Pairs that leave the capacity are told apart by the first launch."""
    ds = tsu.Dataset.generate(500, seed=77, len_min=1000, err_min=0.05)
    for pen in ((5, 6, 2), (4, 6, 2, 24, 1)):
        a = make(tsu, pen[0], [pen[1:3], pen[3:]] if len(pen) > 3 else [pen[1:]])
        try:
            b = a.batch(ds)
            for W in (300, 768):
                got, t = a.align_plain(b, W, raise_on_error=False)
                say(f"{pen} capacity {W}: {int((got < 0).sum())} of 500 overflow, {t['launches']} launches")
                if W == 300 and len(pen) == 3:
                    assert (got < 0).any()
                assert t["launches"] == 1 or (W == 300 and len(pen) > 3)
        finally:
            a.close()
