"""tsu_align_batched_noalloc with penalties other than 4/6/2 at the widest
capacity whose rings fit LDS: pairs whose cells come to the window's edge
without passing it (a gap extension costs 2 or 3, so a pair may end on the
score in between) align, wider ones are refused, as by the ring kernel."""
import ctypes
import random

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
CAPACITY = 4096  # diagonals -2,048 to 2,047; twice as many do not fit LDS


def say(msg):
    print(f"\n[gpu] {msg}", flush=True)


def seq(rng, n):
    return "".join(rng.choice("ACGT") for _ in range(n))


def pair(rng, gap, subs):
    """One gap of `gap` bases at 2,500, substitutions before it."""
    p = seq(rng, 3000)
    t = p
    for i in range(subs):
        at = 1500 + 90 * i
        t = t[:at] + rng.choice([c for c in "ACGT" if c != t[at]]) + t[at + 1:]
    return p, t[:2500] + seq(rng, gap) + t[2500:]


def noalloc(tsu, a, pairs):
    lib = tsu.library()
    words, pr = tsu.Dataset.from_pairs(pairs).packed()
    h = ctypes.c_void_p()
    P = ctypes.POINTER
    r = lib.tsu_batch_create(a._h, words.ctypes.data_as(P(ctypes.c_uint32)), len(words), pr.ctypes.data_as(P(tsu.Pair)),
                             len(pr), ctypes.byref(h))
    assert r == tsu.TSU_OK, tsu.strerror(r)
    b = tsu.Batch(a, h)
    dw, nw, dp, dsc = ctypes.c_void_p(), ctypes.c_int64(), ctypes.c_void_p(), ctypes.c_void_p()
    assert lib.tsu_batch_device(h, ctypes.byref(dw), ctypes.byref(nw), ctypes.byref(dp), ctypes.byref(dsc)) == 0
    scores = np.full(len(pairs), -99, np.int32)
    r = lib.tsu_align_batched_noalloc(a._h, dw, len(words), dp, pr.ctypes.data_as(P(tsu.Pair)), len(pr), dsc,
                                      scores.ctypes.data_as(P(ctypes.c_int32)), None)
    b.close()
    return r, scores


@pytest.mark.parametrize("pen", [(5, 6, 2), (4, 5, 3), (7, 9, 2)])
def test_pairs_that_just_fit(tsu, oracle, pen):
    """Gaps of every length up to the edge and one or two substitutions.  Plain
    form at the same capacity (whose answer is the ring kernel's) says which
    fit."""
    x, o, e = pen
    rng = random.Random(sum(pen))
    pairs = []
    for gap in range(2040, 2048):
        for subs in (0, 1, 2):
            p, t = pair(rng, gap, subs)
            pairs += [(p, t), (t, p)]
    want, _, _ = oracle.wfa_batch(pairs, x, o, e)
    a = tsu.Aligner(x, o, e)
    try:
        a.set_tune_table([{"waves_per_pair": 1, "capacity": CAPACITY, "bucket_bound": 8192}])
        say(f"plain form, {pen}, {len(pairs)} pairs")
        plain, _ = a.align_plain(a.batch(pairs), CAPACITY, raise_on_error=False)
        fit = [q for q, s in zip(pairs, plain) if s >= 0]
        fits = np.array([s for s in plain if s >= 0])
        assert 0 < len(fit) < len(pairs)
        assert (fits == want[plain >= 0]).all()
        say(f"no-allocation form, the {len(fit)} pairs that fit")
        r, got = noalloc(tsu, a, fit)
        assert r == tsu.TSU_OK, a._lib.tsu_last_error(a._h)
        assert (got == fits).all()
        say("no-allocation form, all pairs")
        r, got = noalloc(tsu, a, pairs)
        assert r == tsu.TSU_EKOVERFLOW
        assert (got == plain).all(), np.nonzero(got != plain)[0][:5]
    finally:
        a.close()
