"""The workloads this library's speed is measured on, through its public entry points.

Each case is a dict of plain values: a `form` (the entry point), the pairs and
how they are drawn (count, length range, error range, edit model), penalties
and, for the plain form, the diagonal capacity.  Sizes are the repository's
own workloads (bench.py, tests/) or fractions of them that keep a pass short:
every form, the smallest call that is made in earnest, reads of 100 bp to
60 kbp, 0.5-15% error, gap-affine and 2-piece penalties.

Outputs are whole numbers (scores, CIGAR runs), so they are compared as they
are; `exact` computes the scores of the shortest reads by plain dynamic
programming.
"""
import ctypes
import math
import random

import numpy as np

import tsunami_pact_amd as tsu

PEN = (4, 6, 2)              # the penalties of every named workload
OTHER = (5, 6, 2)            # a set without a common divisor: the general kernel
TWO_PIECE = (4, 6, 2, 24, 1)  # WFA2-lib's default 2-piece set
EDIT_MODES = {"mixed": 0, "substitutions": 1}


def _case(form, pairs, lmin, lmax, emin, emax, name=None, pen="affine", edits="mixed", wf=0):
    c = {"form": form, "pairs": pairs, "len_min": lmin, "len_max": lmax, "err_min": emin, "err_max": emax,
         "penalties": pen, "edits": edits, "wf_length": wf}
    if name:
        c["name"] = name
    return c


def _bound_capacity(length, err):
    """wf_length for the score bound of `length` bases at error rate `err`,
    as the benchmark sizes it: 2 floor((s - o) / e) + 3."""
    x, o, e = PEN
    return 2 * max(0, (int(round(err * length)) * (o + e) - o) // e) + 3


def listed():
    return [
        # short reads against their candidates, one small resident batch per
        # call: launch and copy latency count (bench.py's 100 bp workload)
        _case("plain", 10_000, 100, 100, 0.02, 0.02, "plain_100bp", wf=100),
        # the headline workload at a quarter of its pairs (bench.py: 1,000 bp, 5%)
        _case("plain", 250_000, 1000, 1000, 0.05, 0.05, "plain_1kbp", wf=397),
        # accurate long reads, substitutions only, as in the reference's own
        # grid (10,240 bp at 1%, wf_length 350), at up to that rate
        _case("plain", 10_000, 10_240, 10_240, 0.005, 0.01, "plain_10kbp_1pct", edits="substitutions", wf=350),
        # one capacity for reads of very different lengths, as a user of the
        # plain form has them (1,277 diagonals: several waves per pair)
        _case("plain", 10_000, 200, 2000, 0.01, 0.08, "plain_ragged_2kbp", wf=_bound_capacity(2000, 0.08)),
        # the drop-in path from host characters to scores: packing, copy,
        # alignment (512 bp as in the reference's grid, at up to its 2%)
        _case("fixed", 50_000, 512, 512, 0.005, 0.02, "fixed_512bp", edits="substitutions", wf=42),
        # penalties the register kernels are not built for
        _case("plain", 20_000, 1000, 1000, 0.05, 0.05, "plain_1kbp_other_penalties", pen="other", wf=397),
        # gap-affine 2-piece penalties (bench.py --form twopiece, half its pairs)
        _case("plain", 50_000, 1000, 1000, 0.05, 0.05, "twopiece_1kbp", pen="two_piece", wf=755),
        # mixed reads, batched (bench.py: 100-20,000 bp, 1-15%)
        _case("batched", 30_000, 100, 20_000, 0.01, 0.15, "batched_mixed"),
        # long reads, past the sequence limit of the 16-bit kernels
        _case("batched", 192, 30_000, 60_000, 0.005, 0.02, "batched_60kbp"),
        # CIGARs of long erroneous reads (bench.py: 10,000 bp at 10%)
        _case("cigar", 1_000, 10_000, 10_000, 0.10, 0.10, "cigar_10kbp"),
        # CIGARs of mixed reads
        _case("cigar", 4_000, 100, 10_000, 0.01, 0.15, "cigar_mixed"),
        # a burst of 64 concurrent requests of 1-256 pairs on a running server
        # (bench.py's stream: 100-10,000 bp, 1-15%)
        _case("served", 64, 100, 10_000, 0.01, 0.15, "served_burst"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["plain", "plain", "plain_ragged", "fixed", "other", "two_piece", "batched", "batched", "cigar",
                       "cigar", "served"])
    if kind in ("plain", "plain_ragged", "fixed", "other", "two_piece"):
        top = {"plain": 12_000, "plain_ragged": 4_000, "fixed": 1_100, "other": 1_500, "two_piece": 1_500}[kind]
        L = _log(rng, 60 if kind != "plain_ragged" else 300, top)
        err = rng.uniform(0.005, 0.10 if L <= 3_000 else 0.03)
        lmin = L // rng.randint(2, 8) if kind == "plain_ragged" else L
        edits = "substitutions" if kind == "fixed" else rng.choice(["mixed", "mixed", "substitutions"])
        # about the work of the listed plain cases, never more than the largest
        most = {"plain": 250_000, "plain_ragged": 20_000, "fixed": 60_000, "other": 20_000, "two_piece": 50_000}[kind]
        n = max(33, min(most, int(rng.uniform(0.1, 1.0) * 1.5e8 / (L * (1 + 40 * err * err * L / 100)))))
        if kind in ("other", "two_piece"):
            n = max(33, n // 5)
        pen = {"other": "other", "two_piece": "two_piece"}.get(kind, "affine")
        wf = _bound_capacity(L, err)
        if kind == "two_piece":
            wf = min(2 * wf, 1_900)
        return _case("fixed" if kind == "fixed" else "plain", n, lmin, L, 0.005, err,
                     pen=pen, edits=edits, wf=max(wf, 16))
    if kind == "batched":
        lmax = _log(rng, 500, 20_000)
        lmin = max(50, lmax // rng.choice([1, 3, 20, 200]))
        n = max(50, int(rng.uniform(0.05, 1.0) * 2.0e11 / max(lmax, 2_000) ** 2 / 6))
        return _case("batched", min(n, 20_000), lmin, lmax, 0.01, rng.uniform(0.02, 0.15))
    if kind == "cigar":
        lmax = _log(rng, 500, 10_000)
        lmin = max(50, lmax // rng.choice([1, 3, 20]))
        n = max(20, int(rng.uniform(0.1, 1.0) * 5.0e10 / max(lmax, 4_000) ** 2))
        return _case("cigar", min(n, 3_000), lmin, lmax, 0.01, rng.uniform(0.02, 0.12))
    return _case("served", rng.randint(1, 64), rng.randint(50, 400), _log(rng, 1_000, 10_000), 0.01,
                 rng.uniform(0.03, 0.15))


def _dataset(case, seed, n):
    return tsu.Dataset.generate(n, seed=seed, len_min=case["len_min"], len_max=case["len_max"],
                                err_min=case["err_min"], err_max=case["err_max"], edit_mode=EDIT_MODES[case["edits"]])


def _aligner(case):
    if case["penalties"] == "two_piece":
        x, o1, e1, o2, e2 = TWO_PIECE
        return tsu.Aligner(x, o1, e1, gap_opening2=o2, gap_extension2=e2)
    return tsu.Aligner(*(OTHER if case["penalties"] == "other" else PEN))


class _CigarProgram:
    """A program of the C interface that keeps a batch and reads every
    CIGAR's runs where the library holds them, into one array it keeps."""

    def __init__(self, case, ds):
        lib = self.lib = tsu.library()
        self.ctx, self.batch = ctypes.c_void_p(), ctypes.c_void_p()
        if lib.tsu_create(ctypes.byref(self.ctx), 0, *PEN) != tsu.TSU_OK:
            raise RuntimeError("tsu_create")
        n = self.n = len(ds)
        if lib.tsu_batch_from_dataset(self.ctx, ds._h, 0, n, ctypes.byref(self.batch)) != tsu.TSU_OK:
            raise RuntimeError("tsu_batch_from_dataset")
        vp = ctypes.c_void_p
        self.get = ctypes.CFUNCTYPE(ctypes.c_int, vp, ctypes.c_int64, vp, vp)(("tsu_cigars_get", lib))
        self.where, self.count = np.zeros(n, np.uint64), np.zeros(n, np.int32)
        # two runs per edit at most; over many pairs the mean length counts
        most = n * (2 * int(round(case["err_max"] * case["len_max"])) + 1)
        if most > 4_000_000:
            most = min(most, int(n * (3 * case["err_max"] * _means(case)[0] + 1)))
        self.runs = np.zeros(most, np.uint32)

    def run(self):
        lib, n = self.lib, self.n
        scores, h, t = np.zeros(n, np.int32), ctypes.c_void_p(), tsu.Timing()
        r = lib.tsu_align_cigar(self.ctx, self.batch, scores.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)),
                                ctypes.byref(h), ctypes.byref(t))
        if r != tsu.TSU_OK:
            raise RuntimeError(f"tsu_align_cigar: {lib.tsu_last_error(self.ctx)}")
        w, c, get, handle = self.where.ctypes.data, self.count.ctypes.data, self.get, h.value
        for i in range(n):
            get(handle, i, w + 8 * i, c + 4 * i)
        if int(self.count.sum()) > len(self.runs):
            raise RuntimeError("more runs than two per edit")
        at = self.runs.ctypes.data
        for src, k in zip(self.where.tolist(), self.count.tolist()):
            ctypes.memmove(at, src, 4 * k)
            at += 4 * k
        lib.tsu_cigars_free(h)
        return scores, self.count, self.runs

    def __del__(self):
        self.lib.tsu_batch_free(self.batch)
        self.lib.tsu_destroy(self.ctx)


def prepare(case, seed):
    form, n = case["form"], case["pairs"]
    if form == "cigar":
        return {"form": form, "program": _CigarProgram(case, _dataset(case, seed, n))}
    a = _aligner(case)
    if form == "fixed":
        # characters in the reference's fixed slots, as its reader leaves them
        # (substitutions keep both sequences at the slot's length)
        pairs = _dataset(case, seed, n).pairs()
        pats, txts = [p for p, _ in pairs], [t for _, t in pairs]
        bufs = ["".join(pats).encode(), "".join(txts).encode()]
        return {"form": form, "aligner": a, "bufs": bufs, "n": n, "len": case["len_max"], "wf": case["wf_length"]}
    if form == "served":
        # the same request sizes for every seed, other sequences
        sizes = np.random.default_rng(n).integers(1, 257, n)
        ds = _dataset(case, seed, int(sizes.sum()))
        words, pairs = ds.packed()
        requests, first = [], 0
        for k in sizes:
            pr = pairs[first:first + k].copy()
            lo = int(pr["p_off"][0])
            hi = int(pr["t_off"][-1] + (pr["t_len"][-1] + 15) // 16)
            pr["p_off"] -= lo
            pr["t_off"] -= lo
            requests.append((words[lo:hi], pr))
            first += int(k)
        return {"form": form, "server": tsu.Server(a), "requests": requests}
    ds = _dataset(case, seed, n)
    return {"form": form, "aligner": a, "batch": a.batch(ds), "out": np.zeros(n, np.int32), "wf": case["wf_length"]}


def run(state):
    form = state["form"]
    if form == "plain":
        # a pair wider than the capacity gets a status in its score slot
        return state["aligner"].align_plain(state["batch"], state["wf"], raise_on_error=False, out=state["out"])[0]
    if form == "batched":
        return state["aligner"].align_batched(state["batch"], out=state["out"])[0]
    if form == "cigar":
        return state["program"].run()
    if form == "fixed":
        lib, a = tsu.library(), state["aligner"]
        scores, t = np.zeros(state["n"], np.int32), tsu.Timing()
        lib.tsu_align_fixed(a._h, state["bufs"][0], state["bufs"][1], state["n"], state["len"], state["wf"],
                            scores.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)), ctypes.byref(t))
        return scores
    server = state["server"]
    tickets = [server.submit_packed(w, p) for w, p in state["requests"]]
    results = [server.wait(t, len(p)) for t, (_, p) in zip(tickets, state["requests"])]
    return np.array([r[0] for r in results], np.int32), np.concatenate([r[1] for r in results])


def _means(case):
    """Mean over pairs of the length, and of the squared number of edits."""
    lo, hi = case["len_min"], case["len_max"]
    span = math.log(hi / lo) if hi > lo else 0.0
    length = (hi - lo) / span if span else float(hi)
    square = (hi * hi - lo * lo) / (2 * span) if span else float(hi) * hi
    e0, e1 = case["err_min"], case["err_max"]
    return length, square * (e0 * e0 + e0 * e1 + e1 * e1) / 3


def work(case):
    """Bytes: each packed sequence read once, a score (and, with CIGARs, about
    two runs per edit) written once; the fixed form reads characters.
    Operations: an edit of the generator costs about 3 score steps (after the
    penalties' common divisor; 5 without one), a step s has about 2 s
    diagonals, each 11 integer operations for its three recurrences and 16 for
    one compare of the extension."""
    length, edits2 = _means(case)
    pairs = case["pairs"] * (128.5 if case["form"] == "served" else 1)
    per_base = 1.0 if case["form"] == "fixed" else 0.25
    nbytes = 2 * length * per_base + 4
    if case["form"] == "cigar":
        nbytes += 4 * 2 * length * (case["err_min"] + case["err_max"]) / 2
    steps2 = (3.0 if case["penalties"] == "affine" else 5.0) ** 2 * edits2
    return {"bytes": pairs * nbytes, "flops": pairs * (steps2 + 1) * (11 + 16)}


def exact(case, seed):
    """Gap-affine scores by plain dynamic programming over all pairs at once;
    for reads too long for that, None."""
    if case["form"] != "plain" or case["penalties"] == "two_piece" or case["pairs"] * case["len_max"] ** 2 > 1.5e8:
        return None
    x, o, e = OTHER if case["penalties"] == "other" else PEN
    pairs = _dataset(case, seed, case["pairs"]).pairs()
    n = len(pairs)
    pl = np.array([len(p) for p, _ in pairs])
    tl = np.array([len(t) for _, t in pairs])
    P = np.zeros((pl.max(), n), np.uint8)
    T = np.zeros((tl.max(), n), np.uint8)
    for i, (p, t) in enumerate(pairs):
        P[:len(p), i] = np.frombuffer(p.encode(), np.uint8)
        T[:len(t), i] = np.frombuffer(t.encode(), np.uint8)
    big = np.int64(1) << 40
    out = np.zeros(n, np.int64)
    cols = T.shape[0] + 1
    M = np.zeros((cols, n), np.int64)
    D = np.full((cols, n), big)          # gaps that consume the pattern
    for j in range(1, cols):
        M[j] = o + j * e
    for i in range(P.shape[0] + 1):
        if i:
            diag = M[0].copy()
            M[0] = o + i * e
            D[0] = M[0]
            ins = np.full(n, big)
            for j in range(1, cols):
                D[j] = np.minimum(D[j], M[j] + o) + e
                ins = np.minimum(ins, M[j - 1] + o) + e
                best = np.minimum(np.minimum(D[j], ins), diag + x * (P[i - 1] != T[j - 1]))
                diag = M[j].copy()
                M[j] = best
        done = np.nonzero(pl == i)[0]
        out[done] = M[tl[done], done]
    if case["wf_length"] < 2 * (out.max() // np.gcd.reduce([x, o, e])) + 3:
        return None                       # a pair may leave the capacity: its slot then holds a status
    return out.astype(np.int32)
