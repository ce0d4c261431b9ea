"""Which diagonal capacities hold a pair, restated from the wavefront limits of
the ring kernels: the range a score computes is one wider than its sources on
each gap side, ends without a cell in bounds are trimmed off, and a pair
overflows at the first score whose range leaves the window."""
import numpy as np

NONE = -(1 << 20)


def window(p_len, t_len, W):
    """First and last diagonal of a capacity, and whether each is no bound of
    the alignment."""
    lo = max(-(W // 2), -p_len - 1)
    hi = lo + W - 1
    if hi > t_len + 1:
        hi = t_len + 1
        lo = max(hi - W + 1, -p_len - 1)
    return lo, hi, lo > -p_len - 1, hi < t_len + 1


def run(p, t, pieces, x):
    """(score, ranges by score, cells by score): the range computed at every
    score up to the end (None where there is no source), and per score the
    diagonals of the wavefronts' first and last cells in bounds as
    {name: (lo, hi)} with name M, I0, D0, I1, D1."""
    P, T = len(p), len(t)
    # bases that p[v:] and t[h:] agree on
    same = np.zeros((P + 1, T + 1), np.int64)
    pb, tb = np.frombuffer(p.encode(), np.uint8), np.frombuffer(t.encode(), np.uint8)
    for v in range(P - 1, -1, -1):
        same[v, :T] = np.where(tb == pb[v], same[v + 1, 1:] + 1, 0)
    k = np.arange(-P - 2, T + 3)   # a cell beyond the bounds on each side
    zero = P + 2

    def shifted(w, by):
        """The wavefront's offsets moved by diagonals, NONE from outside."""
        out = np.full(len(k), NONE)
        if w is None:
            return out
        if by > 0:
            out[by:] = w[1][:-by]
        elif by < 0:
            out[:by] = w[1][-by:]
        else:
            out[:] = w[1]
        return out

    def wavefront(h, lo, hi):
        """Trimmed to its cells in bounds, None without one."""
        h = np.where((k >= lo) & (k <= hi), h, NONE)
        ok = np.flatnonzero((h >= 0) & (h <= T) & (h - k >= 0) & (h - k <= P))
        if not len(ok):
            return None
        h[:ok[0]], h[ok[-1] + 1:] = NONE, NONE
        return (int(k[ok[0]]), int(k[ok[-1]])), h

    m0 = np.full(len(k), NONE)
    m0[zero] = same[0, 0]
    waves = {0: {"M": ((0, 0), m0)}}
    ranges, cells = [(0, 0)], [{"M": (0, 0)}]
    if P == T and m0[zero] == T:
        return 0, ranges, cells
    s = 0
    while True:
        s += 1
        mx = waves.get(s - x, {}).get("M")
        los, his, src = [], [], []
        if mx:
            los.append(mx[0][0]); his.append(mx[0][1])
        for i, (o, e) in enumerate(pieces):
            mo, before = waves.get(s - o - e, {}).get("M"), waves.get(s - e, {})
            ie, de = before.get(f"I{i}"), before.get(f"D{i}")
            src.append((mo, ie, de))
            for w, a, b in ((mo, -1, 1), (ie, 1, 1), (de, -1, -1)):
                if w:
                    los.append(w[0][0] + a); his.append(w[0][1] + b)
        waves[s] = {}
        waves.pop(s - 64, None)
        if not los or min(los) > max(his):
            ranges.append(None); cells.append({})
            continue
        lo, hi = min(los), max(his)
        M = shifted(mx, 0) + 1
        for i, (mo, ie, de) in enumerate(src):
            I, D = np.maximum(shifted(mo, 1), shifted(ie, 1)) + 1, np.maximum(shifted(mo, -1), shifted(de, -1))
            waves[s][f"I{i}"], waves[s][f"D{i}"] = wavefront(I, lo, hi), wavefront(D, lo, hi)
            M = np.maximum(M, np.maximum(I, D))
        ok = (k >= lo) & (k <= hi) & (M >= 0) & (M <= T) & (M - k >= 0) & (M - k <= P)
        M = np.where(ok, M + same[np.where(ok, M - k, 0), np.where(ok, M, 0)], NONE)
        waves[s]["M"] = wavefront(M, lo, hi)
        ranges.append((lo, hi))
        cells.append({n: w[0] for n, w in waves[s].items() if w})
        if M[zero + T - P] >= T:
            return s, ranges, cells


def passes(p, t, W, ranges):
    """The range leaves the capacity at some score up to the end."""
    lo, hi, _, _ = window(len(p), len(t), W)
    return any(r and (r[0] < lo or r[1] > hi) for r in ranges[1:])


def touches(p, t, W, cells):
    """A cell in bounds on an edge diagonal at some score before the end."""
    lo, hi, lo_edge, hi_edge = window(len(p), len(t), W)
    return any((lo_edge and c[0] <= lo) or (hi_edge and c[1] >= hi) for w in cells[1:-1] for c in w.values())


def first_pass(p, t, W, pieces, cells):
    """The packed kernel's form of passes(): the score before which the end
    cell must be reached, from the first gap cells seen on the edge diagonals
    (they go on after the extension), or from M[0][0] where diagonal 0 is one."""
    lo, hi, lo_edge, hi_edge = window(len(p), len(t), W)
    best = 1 << 30
    if (lo_edge and lo == 0) or (hi_edge and hi == 0):
        best = min(o + e for o, e in pieces)
    for s, w in enumerate(cells):
        for i, (_, e) in enumerate(pieces):
            if lo_edge and f"D{i}" in w and w[f"D{i}"][0] <= lo:
                best = min(best, s + e)
            if hi_edge and f"I{i}" in w and w[f"I{i}"][1] >= hi:
                best = min(best, s + e)
    return best
