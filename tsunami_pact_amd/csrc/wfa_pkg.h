// wfa_pkg.h -- packed wavefront kernel for any penalties: one gap piece
// (x, o, e) or two (gap of length L: min(o + L e, o2 + L e2)).
//
// The scheme of wfa_pk.h (two diagonals per 32-bit word, chunks of 128
// diagonals that overlap by kPkStep at each end and exchange their copies
// every kPkStep scores, M and I / D maxima taken at the source's diagonal,
// compares of 8 or 16 bases for both cells), with the history in LDS instead
// of registers, since how far back a score reads follows from the penalties:
//   M      max(x, o, o2) slots: score s reads s - x (mismatch) and s - o,
//          s - o2 (for the gap sources below) and overwrites the oldest
//   GI, GD e slots each: max(M[s-o], I[s]) and max(M[s-o], D[s]), the sources
//          of I and D one diagonal away at s + e (read and overwritten in
//          place); the same for the second piece
// A slot holds one word per lane and chunk; a lane only ever reads its own
// column (the shifts are DPP), so the accesses are conflict-free, and the
// same loop serves every penalty set.
//
// NW waves hold a pair, chunk j belongs to wave j mod NW; they meet at two
// barriers per kPkStep scores, around the exchange of the copies.  Scores
// without sources (penalties whose sums leave gaps) are computed like the
// others and come out NULL.
//
// Out-of-bounds I, D and M cells are NULL where they are computed, as in
// wfa_pk.h (the oracle's orc_wfa_nulled: the same scores).  The window is
// that of the ring or 2-piece register kernel it stands in for, and so is the
// answer whether a pair fits it (edges that are bounds of the alignment hold
// nothing):
//   edge_pass  the ring kernels': a pair overflows at the first score whose
//          range leaves the window.  The first cell in bounds on an edge
//          diagonal is a gap's (or M[0][0]), and where GI or GD of s holds one
//          the range goes beyond at s + e: the end must be reached before the
//          least of these (before o + e where diagonal 0 is an edge).
//   else   the 2-piece register kernel's: at the first score with a cell in
//          bounds on an edge diagonal, unless it ends there.  Past probe_cap,
//          that kernel's last score, the ring kernel's answer at the capacity
//          asked for counts; the plain form gives such pairs to it.
//
// What bounds it: instruction issue and LDS reads per chunk and score (45
// vector, 20 scalar and 11 LDS instructions with expanded sequences; 0.89
// vector instructions per CU-cycle at 5/6/2 with packed ones) with one gap
// piece; with two, whose ring is two to four times as large, the
// pairs that fit a CU (vector units 32% busy with two pairs, 4/6/2/24/1).  Copying slot by slot at the exchange took 3.0 ms where
// copying ten slots per LDS instruction takes 2.2 (20,000 x 1,000 bp at 5%,
// 5/6/2, 397 diagonals; now 2.07; the ring kernel 9.2).
#pragma once

#include "wfa_pk.h"

namespace tsu {

constexpr int kPkEvPass = 2;  // the range leaves the window after this score (wfa_pk.h: the other events)
constexpr int kPkgHl = kPkStep / 2;   // lanes of copies at each end
constexpr uint32_t kPkgNone = ~0u;  // a lane that copies nothing
constexpr int kPkgRenull = 8190;  // scores, a multiple of kPkStep: NULL grows by one per score

// Slots of M, and the ring's bytes for a pair.
__host__ __device__ constexpr int pkg_m_slots(int x, int o, int o2) {
    const int a = x > o ? x : o;
    return a > o2 ? a : o2;
}
// The 2-piece kernel with GI and GD in registers: the register kernel's
// extensions and windows, a wave per chunk.
inline bool pkg_in_registers(const Shape& sh) { return sh.two_piece && sh.reg_e && sh.nw == 8 && pkg_chunks(sh.win) <= 8; }
inline int64_t pkg_ring_bytes(const Shape& sh, const KArgs& a) {
    const int64_t m = pkg_m_slots(a.x, a.o, sh.two_piece ? a.o2 : 0), gi = 2ll * a.e + (sh.two_piece ? 2ll * a.e2 : 0);
    return pkg_chunks(sh.win) * (m * 256 + gi * (pkg_in_registers(sh) ? 8 * kPkgHl : 256));
}

// E1, E2 > 0 (two pieces; extensions of 1-3 after the gcd): GI and GD in
// registers, a chunk per wave (NW >= chunks), their slots fixed by unrolling
// the scores of a block; the edges' words go through LDS.  4/6/2/24/1 in 768
// diagonals: 49 KB and three pairs per CU instead of 59 KB and two, six LDS
// instructions a score less; 50,000 x 1,000 bp at 5% 19.2 -> 13.1 ms.
// (Loading the M a score reads during the score before: 13.0, not kept, since
// M must then be two scores old.)
template <int NW, int P, bool H, bool QUEUE, int E1 = 0, int E2 = 0>
__global__ __launch_bounds__(NW * 64) void wfa_pkg_kernel(KArgs a) {
    static_assert(P == 1 || P == 2, "gap pieces");
    constexpr bool RG = E1 > 0;
    static_assert(!RG || (P == 2 && kPkStep % E1 == 0 && kPkStep % E2 == 0), "slots fixed within a block");
    constexpr int EN1 = RG ? E1 : 1, EN2 = RG ? E2 : 1;
    constexpr int NT = NW * 64;
    constexpr int OWN = kPkgOwn, HL = kPkgHl;
    constexpr int XI = 64 / (2 * HL), XR = ((RG ? 1 : 2 * P + 1) * kPkStep + XI - 1) / XI;  // slots copied per round, rounds
    extern __shared__ __align__(16) uint32_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t hn = pk_expanded_entries<H>((uint32_t)a.seq_words);
    const uint32_t hp = pk_expanded_pattern<H>((uint32_t)a.seq_words);
    const uint32_t hpb = 2 * hn;
    const int sw = (int)pk_packed_words((uint32_t)a.seq_words);
    const uint32_t tb = 2 * (hn + hp), pb = tb + 4u * (uint32_t)sw;
    uint32_t* sS = smem + tb / 4;
    int32_t* X = reinterpret_cast<int32_t*>(sS + 2 * sw);  // [0] queue index, [1] first event, [2] edges
    uint32_t* ring = reinterpret_cast<uint32_t*>(X + 4);
    const uint32_t rb = tb + 8u * (uint32_t)sw + 16u;      // its byte address
    const bool lds_at_zero = (uint32_t)(uintptr_t)smem == 0u;
    const int W = a.W;
    const int NC = pkg_chunks(W);
    const uint32_t stride = (uint32_t)NC * 256u;           // bytes per slot
    const int R = pkg_m_slots(a.x, a.o, P == 2 ? a.o2 : 0);
    const int gi1 = R, gd1 = gi1 + a.e, gi2 = gd1 + a.e, gd2 = P == 2 ? gi2 + a.e2 : gi2;
    const int slots = RG ? R : P == 2 ? gd2 + a.e2 : gi2;
    const uint32_t gx = rb + (uint32_t)R * stride;         // RG: the G words exchanged (2 HL per register and chunk)
    const int ahead = max(R, P == 2 ? max(a.e, a.e2) : a.e);
    const uint32_t lane4 = 4u * (uint32_t)lane;

    for (int iter = 0;; ++iter) {
        int idx;
        if constexpr (QUEUE) {
            if (tid == 0) X[0] = atomicAdd(a.queue, 1);
            __syncthreads();
            idx = __builtin_amdgcn_readfirstlane(X[0]);
            __syncthreads();
        } else {
            if (iter > 0) break;
            idx = blockIdx.x;
        }
        if (idx >= a.n) break;
        const int pi = a.order ? __builtin_amdgcn_readfirstlane(a.order[idx]) : idx;
        const KPair pr = a.pairs[pi];
        const int p = __builtin_amdgcn_readfirstlane(pr.p_len);
        const int t = __builtin_amdgcn_readfirstlane(pr.t_len);
        pk_stage(a.words, pr, p, t, sS, sw, tid, NT);
        for (int i = tid; i < slots * NC * 64; i += NT) ring[i] = kPkNull;
        if constexpr (RG) {
            for (int i = tid; i < 2 * (E1 + E2) * NC * 2 * HL; i += NT) pk_st32(gx + 4u * (uint32_t)i, kPkNull);
        }
        if (tid == 0) {
            // the event of a gap cell of piece 1 or 2 on an edge, less 4 s (in
            // LDS: in registers it costs the score loop spills)
            auto then = [&](int scores) -> int { return a.edge_pass ? 4 * (scores - 1) + kPkEvPass : kPkEvEdge; };
            X[1] = W > 2 ? kPkNoEvent : then(P == 2 ? min(a.o + a.e, a.o2 + a.e2) : a.o + a.e);  // (diagonal 0 an edge)
            X[2] = then(a.e) | (P == 2 ? then(a.e2) << 16 : 0);
        }
        __syncthreads();
        if constexpr (H) {
            pk_expand(smem, hn, hp, sS, sw, tid, NT);
            __syncthreads();
        }

        int kmin = max(-(W / 2), -p - 1);
        int kmax = kmin + W - 1;
        if (kmax > t + 1) { kmax = t + 1; kmin = max(kmax - W + 1, -p - 1); }
        const int kb = kmin;
        const int tp = t - p;
        const bool tp_in = tp >= kb && tp - kb < NC * OWN;
        const int jtp = tp_in ? (tp - kb) / OWN : -1, jhe = (kmax - kb) / OWN;
        const bool lo_edge = kmin > -p - 1, hi_edge = kmax < t + 1;
        const int ptp = tp_in ? (tp - kb) % OWN + kPkStep : 0, phi = (kmax - kb) % OWN + kPkStep;
        const int dg = abs(tp);
        const int64_t gap1 = a.o + (int64_t)a.e * dg, gap2 = P == 2 ? a.o2 + (int64_t)a.e2 * dg : gap1;
        const int s_bound = (int)min<int64_t>((int64_t)a.x * min(p, t) + (dg ? min(gap1, gap2) : 0), 0x3fffffff);
        const int dlo = -p - kb, dhi = min(t - kb, OWN * NC - 1), d0 = -kb;

        // score 0: M[0][0] = 0, extended; in every chunk that holds diagonal 0
        const int ext0 = (int)pk_lcp_wave(pb, tb, lane4, 0, 0, min(p, t));
        for (int j = w; j < NC; j += NW) {
            const int k = kb - kPkStep + OWN * j + 2 * lane;
            if (k == 0) ring[j * 64 + lane] = (kPkNull & 0xffff0000u) | (uint32_t)ext0;
            if (k == -1) ring[j * 64 + lane] = (kPkNull & 0xffffu) | ((uint32_t)ext0 << 16);
        }
        // Ring positions (bytes) of the next block's first score, and what a
        // block adds to them.
        const uint32_t Rb = (uint32_t)R * stride, eb = (uint32_t)a.e * stride, eb2 = P == 2 ? (uint32_t)a.e2 * stride : 0u;
        auto next = [&](uint32_t q, uint32_t size) __attribute__((always_inline)) -> uint32_t { q += stride; return q == size ? 0u : q; };
        auto plus = [](uint32_t q, uint32_t n, uint32_t size) __attribute__((always_inline)) -> uint32_t { q += n; return q >= size ? q - size : q; };
        auto start = [&](int s, int depth) -> uint32_t { const int m = s % depth; return (uint32_t)(m < 0 ? m + depth : m) * stride; };
        const uint32_t nR = start(kPkStep, R), ne = start(kPkStep, a.e), ne2 = P == 2 ? start(kPkStep, a.e2) : 0u;
        uint32_t bm = start(1, R), bx = start(1 - a.x, R), bo = start(1 - a.o, R), bg = start(1, a.e);
        uint32_t bo2 = P == 2 ? start(1 - a.o2, R) : 0u, bg2 = P == 2 ? start(1, a.e2) : 0u;
        // The exchange: a lane copies one column of one slot, 60 columns of
        // the 2 kPkgHl times (the kPkStep newest slots of each ring) a round.
        const int col = lane % (2 * HL);
        const int own_lane = col < HL ? col : 64 - 2 * HL + col;      // the copy's lane
        const uint32_t from_lane = (uint32_t)(col < HL ? 64 - 2 * HL + col : col) * 4u;
        const int cM = min(R, kPkStep), c1 = RG ? 0 : min(a.e, kPkStep), c2 = P == 2 && !RG ? min(a.e2, kPkStep) : 0;
        const int items = cM + 2 * c1 + 2 * c2;
        uint32_t xat[XR], xsize[XR], xstep[XR], xbase[XR];  // position in the ring; its size, step and place
#pragma unroll
        for (int u = 0; u < XR; ++u) {
            int q = u * XI + lane / (2 * HL);
            const bool on = lane < XI * 2 * HL && q < items;
            int depth = R, first = 0;
            if (q >= cM) {
                q -= cM;
                depth = a.e; first = gi1;
                if (q >= c1) { q -= c1; first = gd1; }
                if (P == 2 && q >= c1) {
                    q -= c1;
                    depth = a.e2; first = gi2;
                    if (q >= c2) { q -= c2; first = gd2; }
                }
            }
            xat[u] = on ? start(-q, depth) : 0u;  // the slot of s0 - q
            xsize[u] = on ? (uint32_t)depth * stride : ~0u;
            xstep[u] = on ? start(kPkStep, depth) : 0u;
            xbase[u] = rb + (uint32_t)first * stride;
            if (!on) xbase[u] = kPkgNone;
        }
        int g1 = 0, h1 = kPkStep + ahead - a.o, g2 = 0, h2 = P == 2 ? kPkStep + ahead - a.o2 : 0;  // diagonals each piece reaches
        auto reach = [](int& g, int& h, int e) __attribute__((always_inline)) { while (h >= e) { ++g; h -= e; } };
        const PkCompare<H> cmp{tb, pb};
        // RG: slots of GI1, GD1, GI2 and GD2 in turn
        uint32_t G[2 * EN1 + 2 * EN2];
#pragma unroll
        for (uint32_t& v : G) v = kPkNull;
        const bool g_in = lane < HL || lane >= 64 - HL, g_out = (lane >= HL && lane < 2 * HL) || (lane >= 64 - 2 * HL && lane < 64 - HL);
        int s0 = 0, r = 0;
        const bool same = p == t && ext0 == t;
        while (!same) {
            __syncthreads();  // every chunk has its scores up to s0
            const int ev0 = __builtin_amdgcn_readfirstlane(X[1]);
            if ((ev0 >> 2) <= s0) break;
            if (s0 >= s_bound) { r = TSU_EINTERNAL; break; }
            // Diagonals that may hold a cell: a gap opens at o + e and widens
            // the range by one per e scores.  A chunk is computed, and its
            // copies exchanged, from the oldest slot's age before its own
            // diagonals are in that range on: what its copies missed before
            // then leaves the rings before it can reach an own cell.
            reach(g1, h1, a.e);
            h1 += kPkStep;
            if constexpr (P == 2) { reach(g2, h2, a.e2); h2 += kPkStep; }
            const int g = max(g1, g2);
            const int jlo = max(max(d0 - g, dlo), 0) / OWN, jhi = min(d0 + g, dhi) / OWN;
            const int jw = jlo + (w - jlo % NW + NW) % NW;  // this wave's first chunk
            if (s0 > 0) {
                // copies of the neighbours' cells: the kPkStep newest scores
#pragma unroll
                for (int u = 0; u < XR; ++u) xat[u] = plus(xat[u], xstep[u], xsize[u]);
                for (int j = jw; j <= jhi; j += NW) {
                    const int from = col < HL ? j - 1 : j + 1;
                    const bool there = from >= 0 && from < NC;
                    uint32_t v[XR];
#pragma unroll
                    for (int u = 0; u < XR; ++u) {
                        v[u] = kPkNull;
                        if (u * XI < items && xbase[u] != kPkgNone && there) v[u] = pk_ld32(xbase[u] + xat[u] + (uint32_t)from * 256u + from_lane);
                    }
#pragma unroll
                    for (int u = 0; u < XR; ++u)
                        if (u * XI < items && xbase[u] != kPkgNone) pk_st32(xbase[u] + xat[u] + (uint32_t)j * 256u + 4u * (uint32_t)own_lane, v[u]);
                }
                if constexpr (RG) {
                    if (w >= jlo && w <= jhi && g_in) {
                        const int from = lane < HL ? w - 1 : w + 1;
                        const bool there = from >= 0 && from < NC;
                        const uint32_t at = gx + 4u * (uint32_t)(from * 2 * HL + (lane < HL ? HL + lane : lane - (64 - HL)));
#pragma unroll
                        for (int q = 0; q < 2 * (E1 + E2); ++q) {
                            G[q] = kPkNull;
                            if (there) G[q] = pk_ld32(at + (uint32_t)(q * NC * 2 * HL) * 4u);
                        }
                    }
                    if (s0 % kPkgRenull == 0) {
#pragma unroll
                        for (uint32_t& v : G) v = pk_renull(v);
                    }
                }
                if (s0 % kPkgRenull == 0) {
                    for (int j = w; j < NC; j += NW)
                        for (int q = 0; q < slots; ++q) {
                            uint32_t& v = ring[(q * NC + j) * 64 + lane];
                            v = pk_renull(v);
                        }
                }
            }
            __syncthreads();  // copied before any score is overwritten
            int ev = kPkNoEvent;
#pragma unroll 1
            for (int j = jw; j <= jhi; j += NW) {
                const int k = kb - kPkStep + OWN * j + 2 * lane;
                const int l0 = max(min(k + p, t), max(k, 0)), l1 = max(min(k + 1 + p, t), max(k + 1, 0));
                const uint32_t lim = (uint32_t)(l0 & 0xffff) | ((uint32_t)l1 << 16);
                const uint32_t pl = (H ? hpb : 8u * pb) - 2u * (uint32_t)k - 2u;
                const uint32_t A = rb + (uint32_t)j * 256u + lane4;
                const uint32_t A1 = A + Rb, A2 = A1 + 2 * eb;
                // the cells looked at, as thresholds (wfa_pk.h)
                uint32_t watch = 0x7fff7fffu;
                auto cell = [&](int place, int at_least) {
                    const uint32_t sh = 16u * (uint32_t)(place & 1);
                    const uint32_t v = (watch & ~(0xffffu << sh)) | (((uint32_t)(at_least - 1) & 0xffffu) << sh);
                    watch = lane == place >> 1 ? v : watch;
                };
                const bool at_end = j == jtp, at_lo = lo_edge && j == 0, at_hi = hi_edge && j == jhe;
                if (at_end) cell(ptp, t);
                if (at_lo) cell(kPkStep, 0);
                if (at_hi) cell(phi, 0);
                const bool special = at_end || at_lo || at_hi;
                uint32_t qm = bm, qx = bx, qo = bo, qo2 = bo2, qg = bg, qg2 = bg2;
                auto up = [&](uint32_t v) __attribute__((always_inline)) -> uint32_t {
                    const uint32_t u = __builtin_amdgcn_update_dpp(0u, v, 0x138, 0xF, 0xF, true);
                    return pk_add(__builtin_amdgcn_alignbit(v, u, 16), 0x00010001u);
                };
                auto down = [&](uint32_t v) __attribute__((always_inline)) -> uint32_t {
                    const uint32_t u = __builtin_amdgcn_update_dpp(0u, v, 0x130, 0xF, 0xF, true);
                    return __builtin_amdgcn_alignbit(u, v, 16);
                };
                // Score s from the G slots it reads; put() gets their new
                // values, now(i) gives one back (GI1, GD1, GI2, GD2).
                auto score = [&](int s, uint32_t i1, uint32_t d1, uint32_t i2, uint32_t d2, auto put, auto now) __attribute__((always_inline)) {
                    const uint32_t mx = pk_ld32(A + qx), mo = pk_ld32(A + qo);
                    uint32_t mo2 = 0;
                    if constexpr (P == 2) mo2 = pk_ld32(A + qo2);
                    uint32_t I1 = up(i1), D1 = down(d1), I2 = 0, D2 = 0;
                    const uint32_t Xc = pk_add(mx, 0x00010001u);
                    uint32_t M = pk_max(pk_max(D1, Xc), I1);
                    if constexpr (P == 2) {
                        I2 = up(i2);
                        D2 = down(d2);
                        M = pk_max(M, pk_max(I2, D2));
                    }
                    const uint32_t raw = M;
                    if (pk_any(pk_max(M, lim) ^ lim)) {  // a cell out of bounds
                        I1 = pk_null_above(I1, lim);
                        D1 = pk_null_above(D1, lim);
                        M = pk_max(pk_max(D1, Xc), I1);
                        if constexpr (P == 2) {
                            I2 = pk_null_above(I2, lim);
                            D2 = pk_null_above(D2, lim);
                            M = pk_max(M, pk_max(I2, D2));
                        }
                        M = pk_null_above(M, lim);
                    }
                    const uint32_t cl = pk_minu(M, lim);
                    typename PkCompare<H>::Words q;
                    cmp.fetch(cl, pl, q);
                    put(pk_max(mo, I1), pk_max(mo, D1), pk_max(mo2, I2), pk_max(mo2, D2));
                    const uint32_t f = cmp.agree(q);
                    M = pk_add(M, pk_minu(f, pk_sub(lim, cl)));  // (a NULL cell has nothing left)
                    const uint32_t more = f & PkCompare<H>::FULL;
                    if (pk_any(more)) cmp.extend_more(M, lim, more, pl, kb - kPkStep + OWN * j, lane);
                    pk_st32(A + qm, M);
                    if (__builtin_expect(special && pk_any(pk_sub_sat(watch, pk_max(raw, M)) & 0x80008000u), 0)) {
                        auto at = [&](uint32_t v, int place) -> int { return (int16_t)((uint32_t)__builtin_amdgcn_readlane((int)v, place >> 1) >> (16 * (place & 1))); };
                        if (at_end && at(M, ptp) >= t) ev = min(ev, 4 * s + kPkEvEnd);
                        const uint32_t adds = __builtin_amdgcn_readfirstlane((uint32_t)X[2]);
                        auto edge = [&](int place, uint32_t g1, uint32_t g2) {
                            if (at(g1, place) >= 0) ev = min(ev, 4 * s + (int)(adds & 0xffffu));
                            if (P == 2 && at(g2, place) >= 0) ev = min(ev, 4 * s + (int)(adds >> 16));
                        };
                        // M stands for the piece that extends slower (what it
                        // adds is no less than the other's); with W of 1 or 2,
                        // which only queues take, a pair may go wider early
                        if constexpr (RG) {  // (e2 = 1; a chunk has one edge at most)
                            if (at_lo || at_hi) edge(at_lo ? kPkStep : phi, M, at_lo ? now(3) : now(2));
                        } else {
                            if (at_lo) edge(kPkStep, P == 1 ? M : now(1), now(3));
                            if (at_hi) edge(phi, P == 1 ? M : now(0), now(2));
                        }
                    }
                    qm = next(qm, Rb); qx = next(qx, Rb); qo = next(qo, Rb);
                    if constexpr (P == 2) qo2 = next(qo2, Rb);
                };
                if constexpr (RG) {
#pragma unroll
                    for (int i = 1; i <= kPkStep; ++i) {
                        uint32_t &gi = G[i % E1], &gd = G[E1 + i % E1], &gi2r = G[2 * E1 + i % E2], &gd2r = G[2 * E1 + E2 + i % E2];
                        score(s0 + i, gi, gd, gi2r, gd2r, [&](uint32_t ni, uint32_t nd, uint32_t ni2, uint32_t nd2) __attribute__((always_inline)) {
                            gi = ni; gd = nd; gi2r = ni2; gd2r = nd2;
                        }, [&](int i) __attribute__((always_inline)) -> uint32_t { return i == 0 ? gi : i == 1 ? gd : i == 2 ? gi2r : gd2r; });
                    }
                    if (g_out) {
                        const uint32_t at = gx + 4u * (uint32_t)(j * 2 * HL + (lane < 32 ? lane - HL : lane - (64 - 2 * HL) + HL));
#pragma unroll
                        for (int q = 0; q < 2 * (E1 + E2); ++q) pk_st32(at + (uint32_t)(q * NC * 2 * HL) * 4u, G[q]);
                    }
                } else {
#pragma unroll 1
                    for (int s = s0 + 1; s <= s0 + kPkStep; ++s) {
                        const uint32_t ai1 = A1 + qg, ad1 = ai1 + eb, ai2 = A2 + qg2, ad2 = ai2 + eb2;
                        const uint32_t i1 = pk_ld32(ai1), d1 = pk_ld32(ad1);
                        uint32_t i2 = 0, d2 = 0;
                        if constexpr (P == 2) { i2 = pk_ld32(ai2); d2 = pk_ld32(ad2); }
                        score(s, i1, d1, i2, d2, [&](uint32_t ni, uint32_t nd, uint32_t ni2, uint32_t nd2) __attribute__((always_inline)) {
                            pk_st32(ai1, ni);
                            pk_st32(ad1, nd);
                            if constexpr (P == 2) { pk_st32(ai2, ni2); pk_st32(ad2, nd2); }
                        }, [&](int i) __attribute__((always_inline)) -> uint32_t {
                            return P == 1 ? kPkNull : pk_ld32(i == 0 ? ai1 : i == 1 ? ad1 : i == 2 ? ai2 : ad2);
                        });
                        qg = next(qg, eb);
                        if constexpr (P == 2) qg2 = next(qg2, eb2);
                    }
                }
            }
            if (ev != kPkNoEvent) atomicMin(X + 1, ev);
            s0 += kPkStep;
            bm = plus(bm, nR, Rb); bx = plus(bx, nR, Rb); bo = plus(bo, nR, Rb); bg = plus(bg, ne, eb);
            if constexpr (P == 2) { bo2 = plus(bo2, nR, Rb); bg2 = plus(bg2, ne2, eb2); }
        }
        if (tid == 0) {
            const int ev = X[1];
            int score = r;
            if (same) score = 0;
            else if ((ev >> 2) <= s0) {
                score = (ev & 3) == kPkEvEnd ? (ev >> 2) : TSU_EKOVERFLOW;
                if ((ev >> 2) > a.probe_cap) score = QUEUE ? TSU_EKOVERFLOW : kScoreLimit;
            }
            a.scores[pi] = !lds_at_zero ? TSU_EINTERNAL : score < 0 ? score : score * a.g;
        }
        __syncthreads();  // LDS reused by the next pair of this workgroup
    }
}

}  // namespace tsu
