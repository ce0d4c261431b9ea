// wfa_pk.h -- packed wavefront kernel: two diagonals per lane and register.
//
// For the scaled penalties 2/3/1 (4/6/2 and its multiples) and sequences of
// at most 32000 bases.  An offset (0..32000) is exact in 16 bits, so one
// VGPR holds the cells of two neighbouring diagonals and the packed 16-bit
// integer instructions (v_pk_max_i16, v_pk_add_u16, ...) compute both at the
// issue cost of one: the path is bound by vector issue.  Scores are 32-bit.
//
// A chunk is 128 diagonals: lane l holds diagonals 2l (low half) and 2l+1
// (high half).  NW waves of C chunks hold a pair; chunk j belongs to wave
// j mod NW, slot j / NW, so every wave holds an equal share of any range.
//
// Neighbouring chunks overlap.  Of a chunk's 128 diagonals the middle 116
// are its own and kPkStep at each end are copies of its neighbours'.  A cell
// depends on its neighbours one diagonal away one score before, so from exact
// copies a chunk computes kPkStep scores of its own diagonals without a word
// from another chunk; then the chunks exchange the copies, through LDS, or
// within a lone wave from register to register (ds_bpermute, which needs no
// LDS memory).  That costs 10% more cells, and takes away, per chunk and
// score, the exchange of edge values and, per score, the wait of the waves of
// a pair for each other (a pair of 16 waves that met at every score spent
// half its time waiting).
//
// State per chunk, five VGPRs and one bound:
//   Mr[3]  M of the scores s-1, s-2, s-3 (slot s mod 3; the loop over scores
//          is unrolled by 3, so every slot index is a constant)
//   mi     max(M[s-4], I[s-1]), the source of I[s] one diagonal up
//   md     max(M[s-4], D[s-1]), the source of D[s] one diagonal down
// Taking the maximum on the source's own diagonal first leaves one shifted
// value per gap wavefront, and since it is taken at the end of score s-1,
// M[s-4] is not needed any more: no ring in LDS, and I and D themselves are
// never kept.
//
// A score step of a chunk is then
//   I = shift_up(mi) + 1        D = shift_down(md)       X = M[s-2] + 1
//   M = max(D, X, I), extended; mi = max(M[s-3], I); md = max(M[s-3], D)
// where a shift by one diagonal is one DPP wave shift and one v_alignbit.
// M[s] extended is first needed at s+2, so the reads of its extension are in
// flight while the recurrences of s+1 are computed.
//
// NULL is any negative value: -32768, growing by at most kPkDrift per score
// while only NULLs feed it; every kPkRenull scores the registers' negative
// values go back to -32768, so none comes near 0.
// lim holds the last offset in bounds, min(k + p, t); on the diagonals below
// -p and above t that a partly used chunk covers it is max(k, 0), and the
// cells at exactly that offset there never reach a diagonal in bounds (their
// neighbours inside are out of bounds and so NULLed).  Out-of-bounds I and D
// cells are NULLed where they are computed, then M is taken from what is
// left, as in orc_wfa_nulled of the oracle (scores and CIGARs equal the
// trimmed computation's, wfa_gpu.cu:633-719).
//
// The extension compares from M clamped to lim (as unsigned, which also
// turns NULL into lim), so every address is inside the padded sequences, and
// the extended M is clamped to lim again (as signed): no lane is masked.
// With H the sequences are expanded in LDS to one 16-bit word of 8 bases per
// position, so the address of a compare is the offset itself, doubled: 8
// instructions for the two cells against 20 with funnel shifts of the packed
// words, at 4.5 instead of 0.5 bytes of LDS per base of a pair.  The host
// takes H where that leaves enough waves per CU.
//
// What bounds it: vector issue.  A chunk and score takes 29 vector
// instructions for 128 cells where no cell is out of bounds or extends past
// its first compare (37 counted over all of a 1,000 bp pair at 5%: those, the
// exchanges and the setup), where the kernels it replaced took 29-35 for 64;
// with 4 waves per SIMD a CU issues 0.66 vector instructions per cycle
// (16 waves per pair) to 0.83 (8 waves), what is missing being LDS latency.
// Measured, before (32-bit offsets in registers, older M scores in an LDS
// ring, a wait per score) and after: 30,000 pairs of 100-20,000 bp at 1-15%,
// batched, 158 -> 73 ms; 10,000 pairs of up to 2,000 bp in one plain launch
// of 4 waves per pair 1.63 -> 0.63 ms; 250,000 x 1,000 bp at 5% (one wave, 5
// chunks) 7.18 -> 6.29 ms; 10,000 x 10,240 bp at up to 1% 0.71 -> 0.57 ms.
// Without LDS for a lone wave's copies, and with the expanded pattern's
// padding left to the words behind it, a 1,000 bp pair takes 4.8 KB, and 32
// instead of 20 waves share a CU (0.63 vector instructions per cycle before):
// 6.29 -> 5.39 ms; the ragged 2,000 bp pairs 0.735 -> 0.684.
//
// Recurrences, bounds and end tests: wfa_gpu.cu:253-331,610-631.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "wfa_bt.h"

namespace tsu {

using KernelFn = void (*)(KArgs);

constexpr uint32_t kPkNull = 0x80008000u;
constexpr int kPkStep = kPackedStep;  // scores between two exchanges: even, and a multiple of 3
constexpr int kPkDrift = 17;        // 16 bases of a first compare and one of I or X
constexpr int kPkRenull = 128;      // exchanges; copies in LDS are one period behind at most
static_assert(2 * (kPkRenull + 1) * kPkStep * kPkDrift < 32768, "NULL stays negative");
constexpr int kPkWaveExtends = 6;   // cells of a chunk extended by the whole wave in turn rather than by their lanes
constexpr int kPkPadBases = 128;    // positions past a sequence's end that a chunk may address

typedef short pk_s16 __attribute__((ext_vector_type(2)));
typedef unsigned short pk_u16 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_max(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(pk_s16, a), __builtin_bit_cast(pk_s16, b)));
}
__device__ __forceinline__ uint32_t pk_min(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(pk_s16, a), __builtin_bit_cast(pk_s16, b)));
}
__device__ __forceinline__ uint32_t pk_minu(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(pk_u16, a), __builtin_bit_cast(pk_u16, b)));
}
__device__ __forceinline__ uint32_t pk_add(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (pk_u16)(__builtin_bit_cast(pk_u16, a) + __builtin_bit_cast(pk_u16, b)));
}
__device__ __forceinline__ uint32_t pk_sub(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (pk_u16)(__builtin_bit_cast(pk_u16, a) - __builtin_bit_cast(pk_u16, b)));
}
// saturating a - b (signed)
__device__ __forceinline__ uint32_t pk_sub_sat(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(pk_s16, a), __builtin_bit_cast(pk_s16, b)));
}
__device__ __forceinline__ uint32_t pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (pk_u16)(__builtin_bit_cast(pk_u16, a) * __builtin_bit_cast(pk_u16, b)));
}
// a * b + c; b a wave-uniform constant
__device__ __forceinline__ uint32_t pk_mad(uint32_t a, uint32_t b, uint32_t c) {
    uint32_t r;
    asm("v_pk_mad_u16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
}
__device__ __forceinline__ uint32_t pk_half(uint32_t a) {  // each half >> 1
    return __builtin_bit_cast(uint32_t, (pk_u16)(__builtin_bit_cast(pk_u16, a) >> (pk_u16)1));
}
// halves of v above lim (signed) become NULL; a NULL half becomes or stays NULL
__device__ __forceinline__ uint32_t pk_null_above(uint32_t v, uint32_t lim) {
    const pk_s16 m = __builtin_bit_cast(pk_s16, pk_sub(lim, v)) >> (pk_s16)15;
    const uint32_t mm = __builtin_bit_cast(uint32_t, m);
    return (mm & kPkNull) | (~mm & v);
}
// negative halves become NULL
__device__ __forceinline__ uint32_t pk_renull(uint32_t v) {
    const uint32_t mm = __builtin_bit_cast(uint32_t, (pk_s16)(__builtin_bit_cast(pk_s16, v) >> (pk_s16)15));
    return (mm & kPkNull) | (~mm & v);
}
__device__ __forceinline__ int32_t pk_get(uint32_t v, int half) { return (int32_t)(int16_t)(v >> (16 * half)); }

// twice the low / high half of v, zero-extended (SDWA: the select is free)
__device__ __forceinline__ uint32_t pk_lo2(uint32_t v) {
    uint32_t r;
    asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0" : "=v"(r) : "s"(1), "v"(v));
    return r;
}
__device__ __forceinline__ uint32_t pk_hi2(uint32_t v) {
    uint32_t r;
    asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1" : "=v"(r) : "s"(1), "v"(v));
    return r;
}

// (a ^ b) + c in one instruction
__device__ __forceinline__ uint32_t pk_xad(uint32_t a, uint32_t b, uint32_t c) {
    uint32_t r;
    asm("v_xad_u32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
    return r;
}

__device__ __forceinline__ bool pk_any(uint32_t x) { return __builtin_amdgcn_ballot_w64(x != 0u) != 0ull; }

typedef __attribute__((address_space(3))) const uint16_t pk_lds_u16;
typedef __attribute__((address_space(3))) const uint32_t pk_lds_u32;
__device__ __forceinline__ uint32_t pk_ld16(uint32_t a) { return *reinterpret_cast<pk_lds_u16*>((uintptr_t)a); }
__device__ __forceinline__ uint32_t pk_ld32(uint32_t a) { return *reinterpret_cast<pk_lds_u32*>((uintptr_t)a); }
typedef __attribute__((address_space(3))) uint32_t pk_lds_w32;
__device__ __forceinline__ void pk_st32(uint32_t a, uint32_t v) { *reinterpret_cast<pk_lds_w32*>((uintptr_t)a) = v; }

// LDS layout (bytes) of a launch: with H the text's expanded words, then the
// pattern's; then the text's packed words, then the pattern's; then 32-bit
// words for the queue index and the exchange of several waves.  (A cell among the copies may
// hold an offset h < k, whose pattern position h - k is negative but not
// below -t - kPkPadBases: the pattern follows a text at least that long.)
template <bool H>
__host__ __device__ constexpr uint32_t pk_expanded_entries(uint32_t seq_words) {
    // positions 0 .. max_len + kPkPadBases, even (16 * seq_words >= max_len + 32)
    return H ? 16 * seq_words + kPkPadBases - 24 : 0;
}
// The pattern's are fewer: past max_len + 16 a compare reads the words behind
// them, for lanes at a bound, which have nothing left to extend.
template <bool H>
__host__ __device__ constexpr uint32_t pk_expanded_pattern(uint32_t seq_words) { return H ? 16 * seq_words - 16 : 0; }
// (as far as one may read behind them, p + 122 positions)
constexpr int64_t pk_expanded_reach(uint32_t seq_words) { return 2 * (pk_expanded_entries<true>(seq_words) + 16ll * seq_words + kPkPadBases); }
__host__ __device__ constexpr uint32_t pk_packed_words(uint32_t seq_words) { return seq_words + kPkPadBases / 16; }

// LDS bytes of a launch with `state` bytes behind the sequences.
inline int64_t pk_lds_bytes(const Shape& sh, uint32_t sw, int64_t state) {
    const int64_t packed = 8ll * pk_packed_words(sw) + state;
    if (!sh.expand) return packed;
    const int64_t x = 2ll * (pk_expanded_entries<true>(sw) + pk_expanded_pattern<true>(sw)) + packed;
    return x > pk_expanded_reach(sw) ? x : pk_expanded_reach(sw);
}

// Both sequences' packed words into LDS (text at sS, pattern sw words on).
// Past their ends the text holds 1 bits and the pattern 0 bits per base, so a
// compare that starts at a bound seldom matches.
__device__ __forceinline__ void pk_stage(const uint32_t* words, const KPair& pr, int p, int t, uint32_t* sS, int sw, int tid, int nt) {
    const int pw = (p + 15) >> 4, tw = (t + 15) >> 4;
    for (int i = tid; i < sw; i += nt) {
        uint32_t wp = 0u, wt = 0x55555555u;
        if (i < pw) wp = words[pr.p_off + i];
        if (i < tw) wt = words[pr.t_off + i];
        sS[sw + i] = wp;
        if (i == tw - 1 && (t & 15)) wt = (wt & ~(~0u << (2 * (t & 15)))) | (0x55555555u << (2 * (t & 15)));
        sS[i] = wt;
    }
}
// Their expanded words (the text's hn positions at x, the pattern's hp after
// them): two positions per 32-bit word, from a window of 16 bases.
__device__ __forceinline__ void pk_expand(uint32_t* x, uint32_t hn, uint32_t hp, const uint32_t* sS, int sw, int tid, int nt) {
    for (int i = tid; i < (int)hn / 2; i += nt) {
        const int j = i >> 3;
        const uint32_t sh = 4u * (uint32_t)i;
        const uint32_t wt = __builtin_amdgcn_alignbit(sS[j + 1], sS[j], sh);
        const uint32_t wp = __builtin_amdgcn_alignbit(sS[sw + j + 1], sS[sw + j], sh);
        x[i] = (wt & 0xffffu) | ((wt >> 2) << 16);
        if (i < (int)hp / 2) x[hn / 2 + i] = (wp & 0xffffu) | ((wp >> 2) << 16);
    }
}

// Bases that pattern[v..] and text[h..] agree on, at most left, from the
// packed words at LDS bytes pb and tb: all lanes of the wave compare 16 bases
// each, 1,024 at a time.  Arguments and result are the same on every lane
// (but lane4, four times the lane).
__device__ __forceinline__ uint32_t pk_lcp_wave(uint32_t pb, uint32_t tb, uint32_t lane4, int v, uint32_t h, int left) {
    uint32_t n = 0;
    while (left > 0) {
        const uint32_t o = min(lane4, (uint32_t)(left >> 4) << 2);  // lanes past the end repeat its word
        const uint32_t ap = o + (pb + (uint32_t)((v >> 4) * 4)), at = o + (tb + ((h >> 4) << 2));
        const uint32_t x = __builtin_amdgcn_alignbit(pk_ld32(ap + 4), pk_ld32(ap), 2u * (uint32_t)v) ^
                           __builtin_amdgcn_alignbit(pk_ld32(at + 4), pk_ld32(at), 2 * h);
        const uint64_t diff = __builtin_amdgcn_ballot_w64(x != 0);
        if (diff) {
            const int q = __builtin_ctzll(diff);
            return n + (uint32_t)min(left, 16 * q + (__builtin_ctz((uint32_t)__builtin_amdgcn_readlane((int)x, q)) >> 1));
        }
        n += (uint32_t)min(left, 1024);
        h += 1024; v += 1024; left -= 1024;
    }
    return n;
}

// The compares of two cells' extensions.
template <bool H>
struct PkCompare {
    uint32_t tb, pb;  // LDS bytes of the packed text and pattern
    static constexpr uint32_t FULL = H ? 0x00080008u : 0x00100010u;  // a half's compare matched to its end
    // Reads and result apart, so that arithmetic fits between them.
    struct Words {
        uint32_t r[H ? 4 : 8];
        uint32_t s[H ? 1 : 4];
    };
    // The compares from position cl (text) and cl - k (pattern); b: the
    // lane's and chunk's part of the pattern's address for the high half.
    __device__ __forceinline__ void fetch(uint32_t cl, uint32_t b, Words& q) const {
        const uint32_t ha = pk_lo2(cl), hb = pk_hi2(cl);
        const uint32_t va = ha + b, vb = hb + b;  // va is 2 short
        if constexpr (H) {
            q.r[0] = pk_ld16(ha);
            q.r[1] = pk_ld16(va + 2);
            q.r[2] = pk_ld16(hb);
            q.r[3] = pk_ld16(vb);
        } else {
            const uint32_t va2 = va + 2;
            // (the text's words start at LDS 0; an offset doubled is a bit position)
            const uint32_t ap = (va2 >> 3) & ~3u, at = (ha >> 3) & ~3u, bp = (vb >> 3) & ~3u, bt = (hb >> 3) & ~3u;
            q.r[0] = pk_ld32(at); q.r[1] = pk_ld32(at + 4);
            q.r[2] = pk_ld32(ap); q.r[3] = pk_ld32(ap + 4);
            q.r[4] = pk_ld32(bt); q.r[5] = pk_ld32(bt + 4);
            q.r[6] = pk_ld32(bp); q.r[7] = pk_ld32(bp + 4);
            q.s[0] = ha; q.s[1] = va2; q.s[2] = hb; q.s[3] = vb;
        }
    }
    // Bases (at most 8 with H, 16 without) on which the sequences agree.
    __device__ __forceinline__ uint32_t agree(const Words& q) const {
        if constexpr (H) {
            // bit 16 ends a full match
            const uint32_t xa = pk_xad(q.r[0], q.r[1], 0x10000u), xb = pk_xad(q.r[2], q.r[3], 0x10000u);
            return pk_half((uint32_t)__builtin_ctz(xa) | ((uint32_t)__builtin_ctz(xb) << 16));
        } else {
            const uint32_t xa = __builtin_amdgcn_alignbit(q.r[1], q.r[0], q.s[0]) ^ __builtin_amdgcn_alignbit(q.r[3], q.r[2], q.s[1]);
            const uint32_t xb = __builtin_amdgcn_alignbit(q.r[5], q.r[4], q.s[2]) ^ __builtin_amdgcn_alignbit(q.r[7], q.r[6], q.s[3]);
            // (all ones where nothing differs: 0xffff in that half)
            const uint32_t fa = xa ? (uint32_t)__builtin_ctz(xa) : 0xffffffffu;
            const uint32_t fb = xb ? (uint32_t)__builtin_ctz(xb) : 0xffffffffu;
            return pk_minu(pk_half(__builtin_amdgcn_perm(fb, fa, 0x05040100u)), 0x00100010u);
        }
    }
    // Past a full compare, one cell at a time by the whole wave (most steps
    // have one or two such cells, and an accurate read's runs are long).
    // kc: diagonal of the chunk's first lane.
    __device__ __forceinline__ void extend_wave(uint32_t& M, uint32_t lim, int kc, int lane, uint64_t mask, int half) const {
        const int sh = 16 * half;
        while (mask) {
            const int l = __builtin_ctzll(mask);
            mask &= mask - 1;
            const uint32_t h = ((uint32_t)__builtin_amdgcn_readlane((int)M, l) >> sh) & 0xffffu;
            const int left = (int)((((uint32_t)__builtin_amdgcn_readlane((int)lim, l) >> sh) & 0xffffu) - h);
            const uint32_t n = pk_lcp_wave(pb, tb, 4u * (uint32_t)lane, (int)h - (kc + 2 * l + half), h, left);
            M += lane == l ? n << sh : 0u;
        }
    }
    // Cells whose compare matched to its end go on from there: while there
    // are many, all by further compares; then one by one.
    __device__ __forceinline__ void extend_more(uint32_t& M, uint32_t lim, uint32_t more, uint32_t b, int kc, int lane) const {
        uint64_t ml = __builtin_amdgcn_ballot_w64((more & 0xffffu) != 0), mh = __builtin_amdgcn_ballot_w64((more >> 16) != 0);
        while (__builtin_popcountll(ml) + __builtin_popcountll(mh) > kPkWaveExtends) {
            const uint32_t cl = pk_minu(M, lim);
            Words q;
            fetch(cl, b, q);
            const uint32_t e = pk_minu(agree(q), pk_sub(lim, cl));
            M = pk_add(M, e);
            ml = __builtin_amdgcn_ballot_w64((e & FULL & 0xffffu) != 0);
            mh = __builtin_amdgcn_ballot_w64((e & FULL) >> 16 != 0);
        }
        asm volatile("" : "+s"(kc));
        extend_wave(M, lim, kc, lane, ml, 0);
        extend_wave(M, lim, kc, lane, mh, 1);
    }
};

template <int NW, int C>
struct PkLayout {
    static constexpr int NC = NW * C;
    // a window of one chunk has no neighbours: all 128 diagonals are its own
    static constexpr int HALO = NC == 1 ? 0 : kPkStep;
    static constexpr int OWN = 128 - 2 * HALO;        // diagonals per chunk
    static constexpr int HL = HALO / 2;               // lanes of copies at each end
    // [2][5][NC+2][2][HL] by parity of the exchange, state register, chunk
    // (one guard at each end, NULL) and side: the first and the last HALO of
    // the chunk's own diagonals
    static constexpr int XR = (NC + 2) * 2 * HL;      // words per register
    static constexpr int XP = 5 * XR;                 // words per parity
    static constexpr int XCH = 4;
    static constexpr int MISC = 0;                    // [4] queue index
    static constexpr int PG = XCH + (NW > 1 ? 2 * XP : 0);  // [NW] exchanges each wave has finished
    static constexpr int EV = PG + (NW > 1 ? NW : 0); // [1] first event, score * 4 + kind
    static constexpr int LC = EV + 1;                 // [1] long extensions recorded
    static constexpr int WORDS = EV + 4;
};

// Events of a pair, kept as the minimum of score * 4 + kind: the end cell, a
// non-NULL cell at the window's edge, an internal error.  With several waves
// the minimum is in LDS; each wave publishes the exchanges it has finished
// and goes on once both its neighbours (the owners of the chunks beside its
// own) have finished as many, so neighbours are at most one exchange apart,
// which is what the copies, double-buffered by the exchange's parity, need.
// Every wave runs until it has finished the lowest recorded score, so an
// event at a lower score in a slower wave is never missed.  Waits are bounded
// (KArgs::poll_limit); past the bound the pair ends with TSU_EINTERNAL.
constexpr int kPkEvEnd = 0, kPkEvEdge = 1, kPkEvInternal = 3;
constexpr int kPkNoEvent = 0x7fffffff;
constexpr int kPkSpinCap = 1 << 20;

// Backtrace records: 16 bits per cell, one coalesced 256-byte store per chunk
// and score at ((s * NC + j) * 64 + lane) of the workgroup's region.  The
// kernel keeps no I and D, and a cell's sources are maxima taken at their own
// diagonal, so the gap bits sit where the gap comes from:
//   bit 0   M[s][k] before extension is not X (ties M > D > I,
//           common.h:67-77)
//   bit 1   ... and not D either, so I where bit 0 is set as well
//   bit 2   I[s+1][k+1] opens from M[s-3][k] rather than extending I[s][k]
//   bit 3   D[s+1][k-1] opens from M[s-3][k] rather than extending D[s][k]
//   bits 4-15  the extension's length; kPkLong and above: kPkLong, and the
//           length in the list behind the records (score, diagonal, length;
//           packed_long_words).  A walk that needs a length the full list had
//           no room for ends with kLongListFull: another kernel records the pair
// The walk arrives at a cell with its offset after extension, so the length
// gives the offset before.  16 bits per cell are half the record traffic and
// half the state of records that hold the offset itself.
constexpr uint32_t kPkLong = 4095;

// The walk, by all lanes of a wave in step.  It is a chain of dependent
// reads, so the records of 32 scores and 16 diagonals around the current cell
// are loaded at once (four dwords per lane) and read from there until a step
// leaves the block (a mismatch moves 2 scores down a diagonal, a gap 1 or 4
// scores and one diagonal); the block of the next 32 scores on the same
// diagonals is loaded ahead, so its round trip to memory overlaps the steps
// through this one.  Scores are those of the penalties 2/3/1.
template <int NC, int OWN, int HL>
__device__ __forceinline__ int pk_walk(const uint32_t* rec, const uint32_t* longs, int n_longs, int kb, int s_max, int score,
                                       int p, int t, const KArgs& a, int64_t* out_off, int32_t* out_n) {
    const int lane = (int)(threadIdx.x & 63);
    BtWalk w;
    w.need = 2 * (int64_t)(score / 2) + 2;
    unsigned long long b0 = 0;
    if (lane == 0) b0 = atomicAdd(a.runs_used, (unsigned long long)w.need);
    const uint32_t blo = __builtin_amdgcn_readfirstlane((uint32_t)b0);
    const uint32_t bhi = __builtin_amdgcn_readfirstlane((uint32_t)(b0 >> 32));
    w.base = (int64_t)(((uint64_t)bhi << 32) | blo);
    if (w.base + w.need > a.runs_cap) return TSU_ECIGAR;
    w.out = a.runs + w.base;
    w.nr = 0;
    w.cur_op = 4; w.cur_len = 0;
    w.full = false;
    w.writer = lane == 0;
    w.k = t - p; w.off = t; w.ss = score; w.type = 0;
    w.v = p; w.h = t;
    w.x = 2; w.o = 3; w.e = 1;
    int bs = -1, bd = 0, nd = 0;   // the block's top score and first dword; the next block's first dword
    uint32_t blk[4], nxt[4];       // scores bs - lane/8 - 8 i, dword bd + lane%8; the same of bs - 32
    auto load = [&](uint32_t (&x)[4], int ss, int d0) __attribute__((always_inline)) {
        const int q = min(max(d0 + (lane & 7), 0), NC * OWN / 2 - 1);
        const uint32_t* at = rec + (q / (OWN / 2)) * 64 + HL + q % (OWN / 2);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = at[(int64_t)max(ss - 8 * i - (lane >> 3), 1) * NC * 64];
    };
    // the record of score ss (1..score) on diagonal k: false outside the window
    auto record = [&](int ss, int k, uint32_t& r) __attribute__((always_inline)) -> bool {
        const int d = k - kb;
        if (ss < 1 || ss > s_max || d < 0 || d >= NC * OWN) return false;
        const int dw = d >> 1;
        if ((unsigned)(bs - ss) > 31u || (unsigned)(dw - bd) > 7u) {
            if (bs > 0 && (unsigned)(bs - 32 - ss) < 8u && (unsigned)(dw - nd) < 8u) {
                bs -= 32; bd = nd;
#pragma unroll
                for (int i = 0; i < 4; ++i) blk[i] = nxt[i];
            } else {
                bs = ss; bd = dw - 4;
                load(blk, bs, bd);
            }
            nd = dw - 4;
            load(nxt, bs - 32, nd);
        }
        const int row = bs - ss, li = __builtin_amdgcn_readfirstlane(8 * (row & 7) + dw - bd);
        const int q = __builtin_amdgcn_readfirstlane(row >> 3);
        const uint32_t x = q == 0 ? blk[0] : q == 1 ? blk[1] : q == 2 ? blk[2] : blk[3];
        const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)x, li);
        r = (v >> (16 * (d & 1))) & 0xffffu;
        return true;
    };
    while (w.v > 0 && w.h > 0 && w.ss > 0) {
        uint32_t r;
        if (w.type == 0) {
            if (!record(w.ss, w.k, r)) return TSU_EINTERNAL;
            int e = (int)(r >> 4);
            if (e == (int)kPkLong) {
                // 64 entries of the list at a time
                int at = -1;
                for (int i0 = 0; i0 < n_longs && at < 0; i0 += 64) {
                    const int i = i0 + lane;
                    const bool hit = i < n_longs && (int)longs[3 * i] == w.ss && (int)longs[3 * i + 1] == w.k;
                    const uint64_t m = __builtin_amdgcn_ballot_w64(hit);
                    if (m) at = i0 + (int)__builtin_ctzll(m);
                }
                if (at < 0) return kLongListFull;
                e = __builtin_amdgcn_readfirstlane((int)longs[3 * at + 2]);
            }
            w.emit(0, e);
            w.off -= e; w.v = w.off - w.k; w.h = w.off;
            if (w.v < 0 || w.h < 0) return TSU_EINTERNAL;
            if (w.v == 0 || w.h == 0) break;
            if (!(r & 1u)) { w.emit(1, 1); w.ss -= 2; --w.off; --w.v; --w.h; continue; }
            w.type = (r & 2u) ? 1 : 2;
        }
        if (w.type == 1) {
            w.emit(2, 1); --w.k; --w.off;
        } else {
            w.emit(3, 1); ++w.k;
        }
        if (!record(w.ss - 1, w.k, r)) return TSU_EINTERNAL;
        if (r & (w.type == 1 ? 4u : 8u)) { w.ss -= 4; w.type = 0; } else --w.ss;
        w.v = w.off - w.k; w.h = w.off;
    }
    return bt_end(w, out_off, out_n);
}

// Registers for five waves per SIMD: the 9-chunk score kernels would take 99
// (four waves), and 96 cost no spill; 30,000 pairs of 100-20,000 bp, batched,
// 71.8 -> 70.1 ms.  Six (80) spills.  From eight waves on a pair's waves come
// in multiples of two per SIMD.
constexpr int pk_waves_per_simd(int nw, int c, bool h, bool bt) { return c == 9 && h && !bt && nw <= 4 ? 5 : 1; }

// W is the window's width in diagonals as the host counts it (it may be less
// than the chunks hold): the range a pair may use is
// [kmin, kmin + W - 1], kmin = max(-W/2, -p-1), moved down where it would
// pass t + 1; a non-NULL cell on its first or last diagonal (where that is
// no bound of the alignment) ends the pair with TSU_EKOVERFLOW.
template <int NW, int C, bool H, bool QUEUE, bool PROBE = false, bool BT = false>
__global__ __launch_bounds__(NW * 64, pk_waves_per_simd(NW, C, H, BT)) void wfa_pk_kernel(KArgs a) {
    static_assert(NW >= 1 && NW <= 16 && C >= 1 && C <= 16, "at most 16 waves of 16 chunks");
    static_assert(!PROBE || NW == 1, "the probe runs on one wave");
    using L = PkLayout<NW, C>;
    constexpr int NC = NW * C;
    constexpr int NT = NW * 64;
    constexpr int OWN = L::OWN, HALO = L::HALO, HL = L::HL;
    extern __shared__ __align__(16) uint32_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t hn = pk_expanded_entries<H>((uint32_t)a.seq_words);
    const uint32_t hp = pk_expanded_pattern<H>((uint32_t)a.seq_words);
    const uint32_t hpb = 2 * hn;  // pattern's expanded words (the text's start at 0)
    const int sw = (int)pk_packed_words((uint32_t)a.seq_words);
    const uint32_t tb = 2 * (hn + hp);            // packed words: text,
    const uint32_t pb = tb + 4u * (uint32_t)sw;   // pattern
    uint32_t* sS = smem + tb / 4;
    int32_t* X = reinterpret_cast<int32_t*>(sS + 2 * sw);
    const uint32_t xb = tb + 8u * (uint32_t)sw;  // byte address of X
    // LDS addresses are built from 0: the kernel has no static LDS
    const bool lds_at_zero = (uint32_t)(uintptr_t)smem == 0u;
    const int W = a.W;
    const int wl = w == 0 ? NW - 1 : w - 1;  // owner of chunk j-1
    const int wr = w == NW - 1 ? 0 : w + 1;  // owner of chunk j+1
    const int poll_limit = a.poll_limit > 0 ? a.poll_limit : kPkSpinCap;
    uint32_t* rec = nullptr;    // BT: this workgroup's records, then its long extensions
    uint32_t* longs = nullptr;
    if constexpr (BT) {
        rec = a.rec_g + (int64_t)blockIdx.x * a.rec_cap;
        longs = rec + a.rec_cap - packed_long_words(NC);
    }

    for (int iter = 0;; ++iter) {
        int idx;
        if constexpr (QUEUE) {
            if (tid == 0) X[L::MISC] = atomicAdd(a.queue, 1);
            __syncthreads();
            idx = __builtin_amdgcn_readfirstlane(X[L::MISC]);
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
        for (int i = L::XCH + tid; i < L::WORDS; i += NT)
            X[i] = i < L::PG ? (int32_t)kPkNull : i == L::EV ? kPkNoEvent : 0;
        __syncthreads();
        if constexpr (H) {
            pk_expand(smem, hn, hp, sS, sw, tid, NT);
            __syncthreads();
        }

        // the range a pair may use, and the first chunk's first own diagonal:
        // with one wave, diagonal 0 in the middle of a chunk where the window
        // leaves room, so the range grows on both sides at once
        int kmin = max(-(W / 2), -p - 1);
        int kmax = kmin + W - 1;
        if (kmax > t + 1) { kmax = t + 1; kmin = max(kmax - W + 1, -p - 1); }
        int kb = kmin;
        if constexpr (NW == 1 && C > 1) {
            const int c = -OWN / 2 - (kmin < -OWN / 2 ? (-kmin - OWN / 2 + OWN - 1) / OWN * OWN : 0);
            if (c + OWN * C > kmax) kb = c;
        }
        kb = __builtin_amdgcn_readfirstlane(kb);
        const int tp = t - p;
        // a diagonal's chunk bit in its owner wave, its lane and half
        auto chunk_bit = [&](int k) -> uint32_t {
            const int j = (k - kb) / OWN;
            return k >= kb && j < NC && j % NW == w ? 1u << (j / NW) : 0u;
        };
        auto place = [&](int k) -> int { return k >= kb ? (k - kb) % OWN + HALO : 0; };
        const uint32_t endm = __builtin_amdgcn_readfirstlane(chunk_bit(tp));
        const uint32_t lom = __builtin_amdgcn_readfirstlane(kmin > -p - 1 ? chunk_bit(kmin) : 0u);
        const uint32_t him = __builtin_amdgcn_readfirstlane(kmax < t + 1 ? chunk_bit(kmax) : 0u);
        const int ptp = __builtin_amdgcn_readfirstlane(place(tp));
        const int plo = __builtin_amdgcn_readfirstlane(place(kmin));
        const int phi = __builtin_amdgcn_readfirstlane(place(kmax));
        const int64_t bound_u = 2ll * min(p, t) + (p != t ? 3ll + (int64_t)abs(p - t) : 0);
        const int s_bound = (int)min<int64_t>(bound_u, 0x3fffffff);

        uint32_t Mr[3][C], mi[C], md[C], lim[C];
        const int k0 = kb - HALO + OWN * w + 2 * lane;  // this lane's low diagonal in slot 0
#pragma unroll
        for (int c = 0; c < C; ++c) {
            Mr[0][c] = Mr[1][c] = Mr[2][c] = mi[c] = md[c] = kPkNull;
            const int k = k0 + OWN * NW * c;
            const int l0 = max(min(k + p, t), max(k, 0)), l1 = max(min(k + 1 + p, t), max(k + 1, 0));
            lim[c] = (uint32_t)(l0 & 0xffff) | ((uint32_t)l1 << 16);
        }
        // per-lane part of the pattern position of a cell, v = h - k, in the
        // unit of the compare's address: for the low half; the high half's
        // diagonal is one more
        const uint32_t pl = (H ? hpb : 8u * pb) - 2u * (uint32_t)k0 - 2u;
        // this lane's word of the exchange for slot 0: what it copies out
        // (own diagonals at the chunk's ends) or takes in (copies)
        const bool out_lane = HALO > 0 && NW > 1 && ((lane >= HL && lane < 2 * HL) || (lane >= 64 - 2 * HL && lane < 64 - HL));
        const bool in_lane = HALO > 0 && (lane < HL || lane >= 64 - HL);
        uint32_t xl = 0;
        if constexpr (HALO > 0 && NW == 1) {
            xl = 4u * (uint32_t)(lane < 32 ? 64 - 2 * HL + lane : lane - (64 - 2 * HL));  // the copied cell's lane
        } else if constexpr (HALO > 0) {
            int word;  // chunk j's own are at (j + 1) 2 HL
            if (lane < HL) word = w * 2 * HL + HL + lane;                    // the last of j - 1
            else if (lane >= 64 - HL) word = (w + 2) * 2 * HL + lane - (64 - HL);  // the first of j + 1
            else word = (w + 1) * 2 * HL + (lane < 32 ? lane - HL : lane - (64 - 2 * HL) + HL);
            xl = xb + 4u * (uint32_t)(L::XCH + word);
        }

        // A gap can open at s = 4 (from M[0]) and extends by a diagonal per
        // score: WFA2-lib's limits (wfa_gpu.cu:426-468, without trimming)
        // are |k| <= s - 3 from then on, and k = 0 before.  The chunks whose
        // own diagonals meet them (and the alignment's diagonals -p .. t) are
        // computed; once computed, a chunk is computed from then on, and one
        // not yet computed holds NULL.
        const int dlo = -p - kb, dhi = min(t - kb, OWN * NC - 1), d0 = -kb;

        const uint32_t lane4 = 4u * (uint32_t)lane;
        const PkCompare<H> cmp{tb, pb};

        // score 0: M[0][0] = 0, extended
        const int ext0 = (int)pk_lcp_wave(pb, tb, lane4, 0, 0, min(p, t));
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int k = k0 + OWN * NW * c;
            if (k == 0) Mr[0][c] = (kPkNull & 0xffff0000u) | (uint32_t)ext0;
            if (k == -1) Mr[0][c] = (kPkNull & 0xffffu) | ((uint32_t)ext0 << 16);
        }
        if constexpr (NW > 1) __syncthreads();
        int s0 = 0;           // scores finished
        int ev = kPkNoEvent;  // this wave's first event

        // The next kPkStep scores of the chunk in slot CC.
        auto advance = [&](auto CC) __attribute__((always_inline)) {
            constexpr int c = decltype(CC)::value;
            const int u = s0 / kPkStep;
            if constexpr (HALO > 0 && NW > 1) {
                if (s0 > 0 && in_lane) {
                    const uint32_t x = xl + 4u * (uint32_t)(((u & 1) ^ 1) * L::XP + 2 * HL * NW * c);
                    Mr[0][c] = pk_ld32(x);
                    Mr[1][c] = pk_ld32(x + 4u * L::XR);
                    Mr[2][c] = pk_ld32(x + 8u * L::XR);
                    mi[c] = pk_ld32(x + 12u * L::XR);
                    md[c] = pk_ld32(x + 16u * L::XR);
                }
            }
            uint32_t pc = 0u - 2u * (uint32_t)(OWN * NW * c);
            asm volatile("" : "+s"(pc));  // opaque: one scalar operand, not a register per chunk
            const uint32_t b = pl + pc;
            uint32_t em = endm, el = lom, eh = him;  // opaque: scalar bit tests, no predicates kept
            asm volatile("" : "+s"(em), "+s"(el), "+s"(eh));
            const uint32_t special = (em | el | eh) & (1u << c);
            // The cells looked at after every score, as a threshold per half that
            // no other cell exceeds: the end cell at t, or a window edge at 0.
            uint32_t watch = 0x7fff7fffu;
            if (special) {
                auto cell = [&](int place, int at_least) {
                    const uint32_t sh = 16u * (uint32_t)(place & 1);
                    const uint32_t v = (watch & ~(0xffffu << sh)) | (((uint32_t)(at_least - 1) & 0xffffu) << sh);
                    watch = lane == place >> 1 ? v : watch;
                };
                if (em & (1u << c)) cell(ptp, t);
                if (el & (1u << c)) cell(plo, 0);
                if (eh & (1u << c)) cell(phi, 0);
            }
            typename PkCompare<H>::Words q;
            uint32_t flags = 0;  // BT: record bits 0-3 of the score in flight
            uint32_t* rs = nullptr;  // the chunk's records of the next score (uniform)
            if constexpr (BT) rs = rec + ((int64_t)(s0 + 1) * NC + NW * c + w) * 64;
            // the result of score s's compare, and what hangs on the cell
            auto settle = [&](auto PHC, int s) __attribute__((always_inline)) {
                constexpr int PH = decltype(PHC)::value;
                // (a cell never passes lim; a NULL one grows by less than kPkDrift)
                const uint32_t f = cmp.agree(q);
                const uint32_t before = Mr[PH][c];
                uint32_t M = pk_min(pk_add(before, f), lim[c]);
                const uint32_t more = f & PkCompare<H>::FULL;
                uint32_t len = 0;
                if constexpr (BT) len = pk_sub(M, before);
                if (pk_any(more)) {
                    cmp.extend_more(M, lim[c], more, b, kb - HALO + OWN * (NW * c + w), lane);
                    if constexpr (BT) {  // lengths a record does not hold
                        len = pk_minu(pk_sub(M, before), kPkLong * 0x10001u);
                        // (of own diagonals: a copy whose gap source lies beyond
                        // the chunk starts lower and would list a longer one)
                        const bool own = HALO == 0 || (lane >= HL && lane < 64 - HL);
#pragma unroll 1
                        for (int half = 0; half < 2; ++half) {
                            if (!own || ((len >> (16 * half)) & 0xffffu) < kPkLong || pk_get(before, half) < 0) continue;
                            const uint32_t e = (pk_sub(M, before) >> (16 * half)) & 0xffffu;
                            const int i = atomicAdd(X + L::LC, 1);
                            if (i >= packed_long_words(NC) / 3) continue;
                            longs[3 * i] = (uint32_t)s;
                            longs[3 * i + 1] = (uint32_t)(k0 + OWN * NW * c + half);
                            longs[3 * i + 2] = e;
                        }
                    }
                }
                Mr[PH][c] = M;
                if constexpr (BT) {
                    // uniform base and a 32-bit lane offset: no vector address arithmetic
                    asm volatile("" : "+s"(rs));
                    *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(rs) + (uint32_t)lane4) = pk_mad(len, 0x00100010u, flags);
                    rs += NC * 64;
                }
                if (special && pk_any(pk_sub_sat(watch, M) & 0x80008000u)) {
                    auto at = [&](int place) -> int { return (int16_t)((uint32_t)__builtin_amdgcn_readlane((int)M, place >> 1) >> (16 * (place & 1))); };
                    if ((em & (1u << c)) && at(ptp) >= t) ev = min(ev, 4 * s + kPkEvEnd);
                    // a non-NULL cell at a window edge could extend the range beyond it
                    if ((el & (1u << c)) && at(plo) >= 0) ev = min(ev, 4 * s + kPkEvEdge);
                    if ((eh & (1u << c)) && at(phi) >= 0) ev = min(ev, 4 * s + kPkEvEdge);
                }
            };
            // score s (PH = s mod 3), its compare left in flight
            auto score = [&](auto PHC, auto FIRST, int s) __attribute__((always_inline)) {
                constexpr int PH = decltype(PHC)::value;
                constexpr int S2 = (PH + 1) % 3;  // slot of s-2; PH itself holds s-3
                const uint32_t none = NC == 1 ? kPkNull : 0u;  // beyond a chunk's ends (copies, unless it is the only one)
                const uint32_t su = __builtin_amdgcn_update_dpp(none, mi[c], 0x138, 0xF, 0xF, NC > 1);
                const uint32_t sd = __builtin_amdgcn_update_dpp(none, md[c], 0x130, 0xF, 0xF, NC > 1);
                uint32_t I = pk_add(__builtin_amdgcn_alignbit(mi[c], su, 16), 0x00010001u);
                uint32_t D = __builtin_amdgcn_alignbit(sd, md[c], 16);
                const uint32_t Xc = pk_add(Mr[S2][c], 0x00010001u);
                uint32_t M = pk_max(pk_max(D, Xc), I);
                if constexpr (!decltype(FIRST)::value) settle(std::integral_constant<int, (PH + 2) % 3>{}, s - 1);
                if (pk_any(pk_max(M, lim[c]) ^ lim[c])) {  // a cell out of bounds
                    I = pk_null_above(I, lim[c]);
                    D = pk_null_above(D, lim[c]);
                    M = pk_null_above(pk_max(pk_max(D, Xc), I), lim[c]);
                }
                const uint32_t M3 = Mr[PH][c];
                mi[c] = pk_max(M3, I);
                md[c] = pk_max(M3, D);
                Mr[PH][c] = M;
                if constexpr (BT) {
                    constexpr uint32_t one = 0x00010001u;
                    flags = pk_minu(pk_sub(M, Xc), one);
                    flags = pk_mad(pk_minu(pk_sub(M, D), one), 2 * one, flags);
                    flags = pk_mad(pk_minu(pk_sub(mi[c], I), one), 4 * one, flags);
                    flags = pk_mad(pk_minu(pk_sub(md[c], D), one), 8 * one, flags);
                }
                cmp.fetch(pk_minu(M, lim[c]), b, q);
            };
            using P0 = std::integral_constant<int, 0>;
            using P1 = std::integral_constant<int, 1>;
            using P2 = std::integral_constant<int, 2>;
            // the only chunk of a pair is done at its first event
            auto done = [&]() -> bool { return NC == 1 && ev != kPkNoEvent; };
            score(P1{}, std::true_type{}, s0 + 1);
            score(P2{}, std::false_type{}, s0 + 2);
            if (done()) return;
            score(P0{}, std::false_type{}, s0 + 3);
            if (done()) return;
            score(P1{}, std::false_type{}, s0 + 4);
            if (done()) return;
            score(P2{}, std::false_type{}, s0 + 5);
            if (done()) return;
            score(P0{}, std::false_type{}, s0 + 6);
            if (done()) return;
            settle(P0{}, s0 + 6);
            if constexpr (HALO > 0 && NW > 1) {
                if (out_lane) {
                    int32_t* x = X + (xl - xb) / 4u + (u & 1) * L::XP + 2 * HL * NW * c;
                    x[0] = (int32_t)Mr[0][c];
                    x[L::XR] = (int32_t)Mr[1][c];
                    x[2 * L::XR] = (int32_t)Mr[2][c];
                    x[3 * L::XR] = (int32_t)mi[c];
                    x[4 * L::XR] = (int32_t)md[c];
                }
            }
        };
        static_assert(kPkStep == 6, "advance computes six scores");

        const bool same = p == t && ext0 == t;  // identical sequences: score 0
        int r = same ? 1 : 0;
        while (r == 0) {
            if constexpr (NW > 1) {
                const int u = s0 / kPkStep;
                for (int spins = 0;; ++spins) {
                    const int e = __builtin_amdgcn_readfirstlane(
                        __hip_atomic_load(X + L::EV, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                    if ((e >> 2) <= s0) { r = 1; break; }
                    const int g0 = __builtin_amdgcn_readfirstlane(
                        __hip_atomic_load(X + L::PG + wl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                    const int g1 = __builtin_amdgcn_readfirstlane(
                        __hip_atomic_load(X + L::PG + wr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                    if (g0 >= u && g1 >= u) break;
                    if (spins >= poll_limit) {
                        atomicMin(X + L::EV, ((s0 + 1) << 2) | kPkEvInternal);
                        r = TSU_EINTERNAL;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
                if (r != 0) break;
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            }
            // every wave reaches these limits at the same score
            if (s0 >= s_bound) { r = TSU_EINTERNAL; break; }
            if constexpr (BT) {
                if (s0 + kPkStep >= a.step_cap) { r = TSU_ECIGAR; break; }
            }
            if constexpr (PROBE) {
                if (s0 >= a.probe_cap) { r = kProbeStopped; break; }
            }
            if (s0 > 0 && s0 % (kPkRenull * kPkStep) == 0) {
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    Mr[0][c] = pk_renull(Mr[0][c]);
                    Mr[1][c] = pk_renull(Mr[1][c]);
                    Mr[2][c] = pk_renull(Mr[2][c]);
                    mi[c] = pk_renull(mi[c]);
                    md[c] = pk_renull(md[c]);
                }
            }
            uint32_t act = 0;
            {
                const int g = s0 + kPkStep - 3;
                const int jlo = max(max(d0 - g, dlo), 0) / OWN, jhi = min(d0 + g, dhi) / OWN;
                if constexpr (NW == 1) {
                    act = (2u << jhi) - (1u << jlo);
                } else {
                    const int rlo = (jlo + NW - 1 - w) / NW;
                    const int rhi = jhi >= w ? (jhi - w) / NW : -1;
                    if (rlo <= rhi) act = (2u << rhi) - (1u << rlo);
                }
            }
            act = __builtin_amdgcn_readfirstlane(act);
            // one wave: the copies from the neighbour chunks' registers
            auto take = [&](auto CC) __attribute__((always_inline)) {
                constexpr int c = decltype(CC)::value;
                if constexpr (HALO > 0 && NW == 1 && c < C) {
                    if (act & (1u << c)) {
                        auto from = [&](uint32_t (&v)[C]) __attribute__((always_inline)) {
                            const uint32_t lo = c > 0 ? v[c > 0 ? c - 1 : 0] : kPkNull, hi = c + 1 < C ? v[c + 1 < C ? c + 1 : 0] : kPkNull;
                            const uint32_t x = (uint32_t)__builtin_amdgcn_ds_bpermute((int)xl, (int)(lane < 32 ? hi : lo));
                            v[c] = in_lane ? x : v[c];
                        };
                        from(Mr[0]); from(Mr[1]); from(Mr[2]); from(mi); from(md);
                    }
                }
            };
            if (s0 > 0) {
                take(std::integral_constant<int, 0>{}); take(std::integral_constant<int, 1>{});
                take(std::integral_constant<int, 2>{}); take(std::integral_constant<int, 3>{});
                take(std::integral_constant<int, 4>{}); take(std::integral_constant<int, 5>{});
                take(std::integral_constant<int, 6>{}); take(std::integral_constant<int, 7>{});
                take(std::integral_constant<int, 8>{});
            }
            auto sweep = [&](auto CC) __attribute__((always_inline)) {
                if constexpr (decltype(CC)::value < C) {
                    if (act & (1u << decltype(CC)::value)) advance(CC);
                }
            };
            sweep(std::integral_constant<int, 0>{}); sweep(std::integral_constant<int, 1>{});
            sweep(std::integral_constant<int, 2>{}); sweep(std::integral_constant<int, 3>{});
            sweep(std::integral_constant<int, 4>{}); sweep(std::integral_constant<int, 5>{});
            sweep(std::integral_constant<int, 6>{}); sweep(std::integral_constant<int, 7>{});
            sweep(std::integral_constant<int, 8>{}); sweep(std::integral_constant<int, 9>{});
            sweep(std::integral_constant<int, 10>{}); sweep(std::integral_constant<int, 11>{});
            sweep(std::integral_constant<int, 12>{}); sweep(std::integral_constant<int, 13>{});
            s0 += kPkStep;
            if constexpr (NW == 1) {
                if (ev != kPkNoEvent) r = 1;
            } else {
                if (ev != kPkNoEvent) atomicMin(X + L::EV, ev);
                // this wave's copies before its progress
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                if (lane == 0) __hip_atomic_store(X + L::PG + w, s0 / kPkStep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
        if constexpr (NW > 1) {
            __syncthreads();  // every wave has stopped: the first event is final
            ev = __builtin_amdgcn_readfirstlane(X[L::EV]);
        }
        // r < 0 and no event at a score this wave reached: it stopped there
        int score = r;
        if (same) score = 0;
        else if ((ev >> 2) <= s0)
            score = (ev & 3) == kPkEvEnd ? (ev >> 2) : (ev & 3) == kPkEvInternal ? TSU_EINTERNAL : TSU_EKOVERFLOW;
        if constexpr (PROBE) {
            if (r == kProbeStopped) {
                // the furthest h + v = 2h - k of the newest scores
                int far = 0;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const int k = k0 + OWN * c;
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        const int a0 = pk_get(Mr[q][c], 0), a1 = pk_get(Mr[q][c], 1);
                        if (a0 >= 0) far = max(far, 2 * a0 - k);
                        if (a1 >= 0) far = max(far, 2 * a1 - k - 1);
                    }
                }
                for (int d = 32; d > 0; d >>= 1) far = max(far, __shfl_xor(far, d));
                if (lane == 0) a.probe_out[pi] = far;
            }
        }
        if constexpr (BT) {
            __syncthreads();  // every wave's records written
            if (w == 0) {
                int st = !lds_at_zero ? TSU_EINTERNAL : score < 0 ? score : 0;
                int64_t out_off = 0;
                int32_t out_n = 0;
                if (st == 0)
                    st = pk_walk<NC, OWN, HL>(rec, longs, min(__builtin_amdgcn_readfirstlane(X[L::LC]), packed_long_words(NC) / 3), kb,
                                              s0, score, p, t, a, &out_off, &out_n);
                if (lane == 0) {
                    a.run_off[pi] = out_off;
                    a.run_n[pi] = out_n;
                    a.scores[pi] = st ? st : score * a.g;
                }
            }
        } else if (tid == 0)
            a.scores[pi] = !lds_at_zero ? TSU_EINTERNAL : score < 0 ? score : score * a.g;
        __syncthreads();  // LDS reused by the next pair of this workgroup
    }
}

}  // namespace tsu
