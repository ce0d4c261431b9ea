"""Device memory that CIGAR calls hold: within a budget, and not much more than
they need without one."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu
SEED = 0x5453554E
SLACK = 48 << 20  # a call's other buffers, and the allocator's granularity


def say(msg):
    print(f"\n[gpu] {msg}", flush=True)


def used(tsu):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert tsu.library().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0  # the runtime the library loaded
    return total.value - free.value


def check(a, oracle, ds):
    pairs = ds.pairs()
    want, ops, _ = oracle.wfa_batch(pairs, 4, 6, 2, cigar=True)
    got, cig, t = a.align_cigar(a.batch(ds))
    assert (got == want).all()
    bad = [i for i in range(len(pairs)) if cig[i] != oracle.rle(ops[i])]
    assert not bad, bad[:5]
    return t


@pytest.mark.parametrize("n,length,err,budget_mib", [(1, 7000, 0.08, 64), (2, 7000, 0.08, 96), (3, 3000, 0.10, 24),
                                                     (40, 800, 0.25, 16), (60, 800, 0.25, 256)])
def test_records_stay_within_the_budget(tsu, oracle, n, length, err, budget_mib):
    """Few pairs, whose launch keeps room for recording one of them again in
    twice the window (0.25 errors: they do overflow it): that room too is
    within the budget, and state_bytes tells it."""
    ds = tsu.Dataset.generate(n, seed=SEED + length, len_min=length, err_min=err)
    a = tsu.Aligner(4, 6, 2)
    try:
        check(a, oracle, tsu.Dataset.generate(2, seed=SEED, len_min=300, err_min=0.05))  # streams, staging, code
        a.set_cigar_memory(a.CIGAR_AUTO, 0, budget_mib << 20)
        before = used(tsu)
        say(f"{n} pairs of {length} bp, budget {budget_mib} MiB")
        t = check(a, oracle, ds)
        held = used(tsu) - before
        say(f"state {t['state_bytes'] / 2**20:.1f} MiB, held {held / 2**20:.1f} MiB, {t}")
        assert t["record_launches"] + t["checkpoint_launches"] >= 1
        assert t["state_bytes"] <= budget_mib << 20
        assert held <= (budget_mib << 20) + SLACK
    finally:
        a.close()


def test_a_larger_call_grows_to_twice_what_it_needs_at_most(tsu, oracle):
    """A small call, a larger one, the same again: the second adds at most as
    much as is held or missing, the third nothing; set_cigar_memory gives all
    back."""
    small = tsu.Dataset.generate(60, seed=SEED + 1, len_min=1000, err_min=0.1)
    large = tsu.Dataset.generate(120, seed=SEED + 2, len_min=3000, err_min=0.1)
    a = tsu.Aligner(4, 6, 2)
    try:
        before = used(tsu)
        t1 = check(a, oracle, small)
        first = used(tsu) - before
        t2 = check(a, oracle, large)
        second = used(tsu) - before
        say(f"held {first / 2**30:.2f} GiB, then {second / 2**30:.2f}; states {t1['state_bytes']}, {t2['state_bytes']}")
        need = t2["state_bytes"] * t2["record_launches"]
        assert second <= 2 * max(first, need) + SLACK
        check(a, oracle, large)
        assert used(tsu) - before <= second + SLACK
        a.set_cigar_memory()
        assert used(tsu) - before <= SLACK + (64 << 20)
    finally:
        a.close()
