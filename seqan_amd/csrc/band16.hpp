// band16.hpp -- packed int16 banded scores, one pair couple per lane, global
// under every AlignConfig and local, for gfx950.  Instantiated per DNA profile
// / substitution table and kind by band16.hip.
//
// Banded DP: only the cells with lower <= j - i <= upper exist (the
// reference's banded globalAlignmentScore, include/seqan/align/
// global_alignment_banded.h:152-181, and localAlignmentScore,
// local_alignment_banded.h:242-259, whose band walks dp_algorithm_impl.h's
// banded tracks; every value comes from cells inside the band).  The
// recurrence is the score kernels' (score16.hpp):
//   global, values drifted by d (i + j):
//     E = max(E, G); F = max(F, G); H = max3(D, E, F); G = H - cost; D' = G + t
//   local, values drifted by d (column), rebased every kRebase columns:
//     E = max3(E, G, z); F = max(F, G) - d; H = max3(D, E, F); G = H - cost
// with the bias raised by what the band can cost (bandDrop, engine.cpp).
//
// Every lane holds a couple of pairs (the 16-bit halves of its registers) and
// a wavefront 128 pairs of one length m, so that their rows line up: the
// wavefront sweeps blocks of R rows, bottom-aligned (row m is the last row
// of the last block).  A block of rows i0 .. i0 + R - 1 sweeps only the
// columns its band covers, i0 + lower .. i0 + R - 1 + upper: W - 1 + R
// columns for a band of W diagonals.  Cells outside the band are computed
// like the others but never reach a cell inside it: a cell on the lower
// diagonal (j - i = lower) takes E = -inf (its left neighbour lies outside;
// local: the floor), one on the upper diagonal (j - i = upper) takes F = -inf
// (its upper neighbour lies outside), and a diagonal step stays on its
// diagonal.  Those two boundaries cross the block only in its first and last
// R columns: there row k is forced when k >= u (E; u = j - i0 - lower) or k <=
// u - (W - 1) (F), one bit-select per row with a wavefront-uniform mask (the
// masks depend on k minus the column's place in its group only, so a group
// makes them once); the columns between are plain sweeps.  Both halves of a
// register are outside at once, so whatever the cells outside hold (wrapped
// sums included) stays there.  Row buffer entries a block reads outside the
// columns the block above wrote only feed cells outside the band.
//
// What bounds it: two waves per SIMD (8 waves per CU, whose rings fill the LDS),
// which use 73% of the vector issue slots on the first call below and 57% on
// the second (two rounds of items); an item's blocks in small calls.  1,048,576
// pairs of 150 bp, band [-16, 16], global: 1.62 ms in plain saturating values
// (9 instructions per packed cell, 6.4 now), 1.37 in drifted ones with a wave per
// item, 1.12 with two waves sharing one; 65,536 pairs of 1 kbp, band [-100,
// 100], free ends: 51.8 (a wave per pair in 32 bits) -> 4.0 -> 2.4 ms, 1,000 of
// them 0.81.
#pragma once

#include <type_traits>

#include "kernels.hpp"
#include "packed16.hpp"
#include "seqan_amd.h"

namespace sqmi {
namespace {

constexpr int kBandRebase = 16;   // local: columns between rebases of the drift

// LR: the row-buffer ring lives in LDS (dynamic shared memory) and the waves of
// a workgroup share an item: wave w takes its blocks w, w + waves, ..., each a few
// columns behind the block above, whose progress it reads from LDS (all waves
// of a workgroup run, and block b waits for block b - 1 only, so every wait
// ends; it is bounded besides).  Otherwise each wave has a ring in global
// memory and sweeps items of its own.  WIDE: values above kDriftNarrowMax.
template <int R, bool DNA, int KIND, bool WIDE, bool LR>
struct Band16 {
    static constexpr int QD = 4;   // columns per group: one dword of residues per pair
    static constexpr bool LOC = KIND == kBandLocal, FREE = KIND == kBandFree;

    struct Couple {
        const uint8_t *h[2];
        const uint8_t *v[2];
        int n[2], pid[2];
    };
    struct Best {
        int2 H;            // global: the best tracked cell (H)
        uint32_t b2;       // local: the best G, without drift
    };
    // LR: columns finished, block << 16 | column (0xffff: all), of the wave
    // that sweeps the block above and of this one.
    struct Progress {
        uint32_t *up, *own;
        uint32_t upBase, ownBase;
        uint32_t *error;
        __device__ __forceinline__ void waitFor(int col, uint32_t &seen) const
        {
            const uint32_t need = upBase + (uint32_t)min(col, 0xffff);
            for (int spins = 0; seen < need; ++spins) {
                seen = (uint32_t)__builtin_amdgcn_readfirstlane(
                    (int)__hip_atomic_load(up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                if (seen >= need)
                    break;
                if (spins > (1 << 22)) {
                    __hip_atomic_store(error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    seen = 0xffffffffu;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            asm volatile("" ::: "memory");   // the ring reads stay behind (a wave's LDS operations run in order)
        }
        __device__ __forceinline__ void publish(int col) const
        {
            asm volatile("" ::: "memory");
            __hip_atomic_store(own, ownBase + (uint32_t)col, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    };

    __device__ __forceinline__ static uint32_t add(uint32_t a, uint32_t b) { return WIDE ? uadd2(a, b) : a + b; }
    __device__ __forceinline__ static uint32_t sub(uint32_t a, uint32_t b) { return WIDE ? usub2(a, b) : a - b; }
    __device__ __forceinline__ static uint32_t max3(uint32_t a, uint32_t b, uint32_t c)
    {
        return WIDE ? umax2(umax2(a, b), c) : max3Pos(a, b, c);
    }

    // Residues of a pair as aligned dwords: columns j .. j + 3 are the funnel
    // shift by (j - 1 + mis) % 4 of dwords (j - 1 + mis) / 4 and the next,
    // both clamped to the dword of the pair's last residue (bytes past n are
    // arbitrary: a column never feeds the columns left of it, and results are
    // taken from columns up to n only).
    struct Residues {
        const uint32_t *words;
        uint32_t mis;
        int lastW;
    };
    __device__ __forceinline__ static Residues residues(const uint8_t *h, int n)
    {
        const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(h) & 3u);
        return Residues{reinterpret_cast<const uint32_t *>(h - mis), mis, (int)((max(n, 1) - 1 + (int)mis) >> 2)};
    }

    // One block, rows i0 .. i0 + R - 1 (both pairs of every lane share them).
    // Free first row: the rows above row 0 and row 0 itself hold H = 0, the
    // first block's row above starts it and their score (padScore) keeps it.
    __device__ __forceinline__ static void block(const FwdArgs &a, const Couple &c, int i0, int maxN, int minN, bool first,
                                                 bool last, uint2 *rb, const uint32_t *sProf, const int16_t *sT,
                                                 Best &best, const Progress &pg)
    {
        Drift dr = a.drift;
        dr.d = __builtin_amdgcn_readfirstlane(dr.d);
        dr.cost = __builtin_amdgcn_readfirstlane(dr.cost);
        dr.neg = __builtin_amdgcn_readfirstlane(dr.neg);
        dr.bias = __builtin_amdgcn_readfirstlane(dr.bias);
        const bool leftFree = (a.mode & SQMI_FREE_LEFT) != 0, topFree = (a.mode & SQMI_FREE_TOP) != 0;
        const bool rightFree = FREE && (a.mode & SQMI_FREE_RIGHT) != 0;
        const bool bottomFree = FREE && (a.mode & SQMI_FREE_BOTTOM) != 0;
        const int PAD = a.alpha;
        const int TW = a.alpha + 1;
        const int m = i0 + R - 1;                    // last block: row m
        const int W1 = a.bandUp - a.bandLo;          // W - 1
        const int jS = i0 + a.bandLo;                // the block's first band column (u = 0)
        // Sweep start: the first band column (LDS rings), else rounded down
        // to a multiple of QD plus one (measured faster with global rings).
        const int jA = jS <= 1 ? 1 : LR ? jS : ((jS - 1) & ~(QD - 1)) + 1;
        const int jE = min(i0 + R - 1 + a.bandUp, maxN);           // the block's last band column
        const int jEnd = LR ? jE : (jE + QD - 1) / QD * QD;   // the last group may run past it
        // In vector registers: 32-bit operations with a scalar operand issue
        // at half the rate.
        uint32_t neg2 = (uint32_t)dr.neg * 0x10001u, cost2 = (uint32_t)dr.cost * 0x10001u, d2 = (uint32_t)dr.d * 0x10001u;
        asm volatile("" : "+v"(neg2), "+v"(cost2), "+v"(d2));

        // Per row: DNA the row words of both pairs, else the two row codes;
        // G and E of the column left of the sweep: column 0's border when the
        // sweep starts at column 1, else cells outside the band (-inf).
        uint32_t rowA[R], rowB[DNA ? R : 1];
        uint32_t Gk[R], Ek[R];
        // The rows' residues, all loads first (an empty lane reads the set's
        // first residue; rows above row 1 are padding): one wait per block.
        int raw[R][2];
        if (i0 >= 1) {
            // Rows i0 .. i0 + R - 1 read bytes i0 - 1 .. i0 + R - 2: R / 4 + 1
            // aligned dwords per pair (the last one clamped to the dword of
            // the last byte needed), funnel-shifted into place.
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const uint8_t *p = c.v[x] + (i0 - 1);
                const uint32_t mv = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 3u);
                const uint32_t *w = reinterpret_cast<const uint32_t *>(p - mv);
                uint32_t wv[R / 4 + 1];
#pragma unroll
                for (int q = 0; q < R / 4; ++q)
                    wv[q] = w[q];
                wv[R / 4] = w[min(R / 4, (int)((mv + R - 1) >> 2))];
#pragma unroll
                for (int q = 0; q < R / 4; ++q) {
                    const uint32_t al = __builtin_amdgcn_alignbyte(wv[q + 1], wv[q], mv);
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        raw[4 * q + b][x] = (int)((al >> (8 * b)) & 0xffu);
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < R; ++k) {
#pragma unroll
                for (int x = 0; x < 2; ++x)
                    raw[k][x] = c.v[x][max(i0 + k - 1, 0)];
            }
        }
        const int border = leftFree ? dr.bias - dr.cost : dr.bias - 2 * dr.cost;   // G(i, 0), i >= 1, less
        const int slope = leftFree ? dr.d : 0;                                      // slope * i
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int i = i0 + k;
            int code[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int pad = (i >= 1 && c.pid[x] >= 0) ? 0 : 0xff;   // min() turns 0xff into PAD
                code[x] = min(raw[k][x] | pad, PAD);
            }
            int g0 = dr.neg;
            if (!LOC && jA == 1)
                g0 = i >= 1 ? border + slope * i : i == 0 || topFree ? dr.bias - dr.cost : dr.neg;
            if constexpr (DNA) {
                rowA[k] = sProf[8 + code[0]];
                rowB[k] = sProf[8 + code[1]];
            } else {
                rowA[k] = (uint32_t)code[0] | ((uint32_t)code[1] << 16);
            }
            Gk[k] = (uint32_t)g0 * 0x10001u;
            Ek[k] = neg2;
        }
        if (FREE && last && bottomFree && a.bandLo <= -m) {   // cell (m, 0)
            const int g = (int)(Gk[R - 1] & 0xffffu) + dr.cost - dr.bias - dr.d * m;
            best.H = make_int2(max(best.H.x, g), max(best.H.y, g));
        }
        // The row buffer is a ring of a.bandCols columns (a power of two of at
        // least W - 1 + R + 10): the columns a block uses, jA - 1 to the end
        // of its last group, span at most W + R + 3 (first band column
        // start) or W + R + 6 (group-aligned start) columns, so no column the
        // block writes shares a slot with one it still has to read.
        // The diagonal input of the first swept column, and column 0 of this
        // block's bottom row for the next block.
        const int cm = a.bandCols - 1;
        uint32_t seen = 0;
        if (LR && !first)
            pg.waitFor(jA + QD - 1, seen);
        uint32_t topG = !LOC && topFree ? (uint32_t)(dr.bias - dr.cost) * 0x10001u : neg2;   // first block: G above
        const uint32_t topStep = !LOC && topFree ? d2 : 0u;
        uint32_t upGprev = first ? topG : rb[((jA - 1) & cm) * 64].x;
        if (!last && jA == 1)
            rb[0] = make_uint2(Gk[R - 1], neg2);

        const s16x2 nHalf = pack(c.n[0], c.n[1]);
        uint2 rq[QD];
#pragma unroll
        for (int u = 0; u < QD; ++u)
            rq[u] = first ? make_uint2(neg2, neg2) : rb[((jA + u) & cm) * 64];
        const Residues ra = residues(c.h[0], c.n[0]), rbs = residues(c.h[1], c.n[1]);
        // Column jA is byte jA - 1 of a pair's residues: dword (jA - 1 + mis)
        // / 4 of its aligned words, at byte (jA - 1 + mis) % 4.  With LDS rings
        // (any start) that is a per-lane base wA and shift; otherwise jA - 1 is
        // a multiple of QD and the dword index is the uniform group count gS
        // (the per-lane base measured 6 % slower there).
        const int offA = jA - 1 + (int)ra.mis, offB = jA - 1 + (int)rbs.mis;
        const int wA = LR ? offA >> 2 : 0, wB = LR ? offB >> 2 : 0;
        const int gS = LR ? 0 : (jA - 1) / QD;
        const uint32_t shA = LR ? (uint32_t)offA & 3u : ra.mis, shB = LR ? (uint32_t)offB & 3u : rbs.mis;
        uint32_t a0 = ra.words[min(wA + gS, ra.lastW)], a1 = ra.words[min(wA + gS + 1, ra.lastW)];
        uint32_t b0 = rbs.words[min(wB + gS, rbs.lastW)], b1 = rbs.words[min(wB + gS + 1, rbs.lastW)];

        // The first block reads -inf (or the free row) for the row above; its row-buffer loads
        // still run (in bounds, the values unused), so that no branch splits
        // the column loop, and the choice is made where an entry is used.
        const uint32_t above = first ? 0u : 0xffffffffu;
        uint32_t z2 = (uint32_t)dr.bias * 0x10001u;   // local: the stored 0 at the current drift
        uint32_t b2 = best.b2;                        // local: the best G at the current drift
        int dcol = 0;                                 // local: the columns of the current drift
        // One group of QD columns from s0; EDGE: the group meets a band
        // boundary (some column with u < R or u >= W - 1).
        // The next group's row-buffer entries are read at the start of a
        // group and the group's bottom-row entries stored at its end, so that
        // waiting for a group's loads (vmcnt counts loads and stores in
        // order) never waits for stores issued just before them.
        auto group = [&](auto edge, int s0, uint32_t curA, uint32_t curB) {
            constexpr bool EDGE = decltype(edge)::value;
            uint2 nx[QD], outv[QD];
            // Row k of column s0 + u is forced by a wave-uniform condition on
            // c = k - u alone: one mask per c and boundary for the group
            // (entry c + QD; local: with one more on each side, the masks of the
            // cells outside).
            constexpr int NC = EDGE ? QD + R + 1 : 1;
            uint32_t fE[NC], fF[NC];
            if constexpr (EDGE) {
                const int d0 = s0 - jS;
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    fE[c] = (c - QD >= d0) ? 0xffffffffu : 0u;        // k >= u + d0: j - i <= lower
                    fF[c] = (c - QD <= d0 - W1) ? 0xffffffffu : 0u;   // k <= u + d0 - (W - 1): j - i >= upper
                }
            }
            if constexpr (LOC) {
                if (dcol == kBandRebase) {
                    const uint32_t r = d2 * kBandRebase;
#pragma unroll
                    for (int k = 0; k < R; ++k) {
                        Gk[k] = sub(Gk[k], r);
                        Ek[k] = sub(Ek[k], r);
                    }
                    upGprev = sub(upGprev, r);
                    z2 = sub(z2, r);
                    b2 = sub(b2, r);
                    dcol = 0;
                }
            }
            if (LR && !first)
                pg.waitFor(s0 + 2 * QD - 1, seen);
#pragma unroll
            for (int u = 0; u < QD; ++u)
                nx[u] = rb[((s0 + QD + u) & cm) * 64];   // read before this block writes them, next group
#pragma unroll
            for (int u = 0; u < QD; ++u) {
                const int j = s0 + u;
                topG = add(topG, topStep);
                uint2 up = make_uint2(bfi(above, rq[u].x, topG), bfi(above, rq[u].y, neg2));
                uint32_t lift = 0;
                if constexpr (LOC) {
                    // Row entries carry no drift.
                    lift = (uint32_t)(dcol + u + 1) * (uint32_t)dr.d * 0x10001u;
                    up.x = add(up.x, lift);
                    up.y = add(up.y, lift);
                    z2 = add(z2, d2);
                    b2 = add(b2, d2);
                }
                uint32_t colSel = 0, pA = 0, pB = 0;
                if constexpr (DNA) {
                    // [h_A, 0x0c, h_B + 4, 0x0c]: byte h_A of the pair-A row
                    // word, byte h_B of the pair-B one, zero high bytes.
                    const uint32_t pick = (uint32_t)u | (0x0cu << 8) | ((uint32_t)(4 + u) << 16) | (0x0cu << 24);
                    colSel = (__builtin_amdgcn_perm(curB, curA, pick) & 0x00030003u) | 0x0c040c00u;
                } else {
                    const uint32_t after = asu((nHalf - splat(j)) >> splat(15));   // 0xffff where j > n
                    const int rA = (int)((curA >> (8 * u)) & 0xffu), rB = (int)((curB >> (8 * u)) & 0xffu);
                    pA = (uint32_t)(((after & 0xffffu) ? PAD : min(rA, PAD)) * TW);
                    pB = (uint32_t)(((after >> 16) ? PAD : min(rB, PAD)) * TW);
                }
                auto tOf = [&](int k) -> uint32_t {
                    if constexpr (DNA) {
                        return __builtin_amdgcn_perm(rowB[k], rowA[k], colSel);
                    } else {
                        const uint32_t lo = (uint16_t)sT[(int)pA + (int)(rowA[k] & 0xffffu)];
                        const uint32_t hi = (uint16_t)sT[(int)pB + (int)(rowA[k] >> 16)];
                        return lo | (hi << 16);
                    }
                };
                const uint32_t noF = LOC ? sub(z2, cost2) : neg2;   // F of a cell whose upper neighbour lies outside
                uint32_t uG = up.x, uF = up.y, m2 = 0;
                const uint32_t upG = uG;
                uint32_t D = add(upGprev, tOf(0));
#pragma unroll
                for (int k = 0; k < R; ++k) {
                    uint32_t E = LOC ? max3(Ek[k], Gk[k], z2) : umax2(Ek[k], Gk[k]);
                    uint32_t F = umax2(uF, uG);
                    if constexpr (LOC)
                        F = sub(F, d2);
                    if constexpr (EDGE) {
                        E = bfi(fE[k - u + QD], LOC ? z2 : neg2, E);
                        F = bfi(fF[k - u + QD], noF, F);
                    }
                    Ek[k] = E;
                    const uint32_t H = max3(D, E, F);
                    if (k + 1 < R)
                        D = add(Gk[k], tOf(k + 1));
                    Gk[k] = sub(H, cost2);
                    uG = Gk[k];
                    uF = F;
                    if constexpr (LOC) {
                        // The column's best cell inside the band.
                        if constexpr (EDGE)
                            m2 = umax2(m2, uG & ~(fE[k - u + QD - 1] | fF[k - u + QD + 1]));
                        else if (k % 2 == 1)
                            m2 = k == 1 ? umax2(Gk[0], uG) : max3(m2, Gk[k - 1], uG);
                        else if (k == R - 1)
                            m2 = umax2(m2, uG);
                    }
                }
                upGprev = upG;
                if constexpr (LOC) {
                    const uint32_t in = ~asu((nHalf - splat(j)) >> splat(15));   // 0xffff where j <= n
                    b2 = umax2(b2, m2 & in);
                    outv[u] = make_uint2(sub(uG, lift), sub(uF, lift));
                } else {
                    outv[u] = make_uint2(uG, uF);
                    // Row m: cell (m, n), or every cell inside the band.
                    if (last) {
                        const int off = dr.cost - dr.bias - dr.d * (m + j);
                        const int gA = (int)(uG & 0xffffu) + off, gB = (int)(uG >> 16) + off;
                        const bool in = bottomFree && j - m >= a.bandLo && j - m <= a.bandUp;
                        best.H.x = (j == c.n[0] || (in && j < c.n[0])) ? max(best.H.x, gA) : best.H.x;
                        best.H.y = (j == c.n[1] || (in && j < c.n[1])) ? max(best.H.y, gB) : best.H.y;
                    }
                    if constexpr (FREE) {
                        // Column n: rows kLo .. kHi lie inside the band and
                        // the matrix; going down, the running maximum gains
                        // the drift, so that it compares with the next row.
                        if (rightFree && j >= minN && __any(j == c.n[0] || j == c.n[1])) {
                            const int kLo = max(-i0, j - a.bandUp - i0), kHi = min(R - 1, j - a.bandLo - i0);
                            uint32_t mx = 0;
#pragma unroll
                            for (int k = 0; k < R; ++k) {
                                mx = uadd2(mx, k > kLo ? d2 : 0u);
                                mx = umax2(mx, k >= kLo && k <= kHi ? Gk[k] : 0u);
                            }
                            const int off = dr.cost - dr.bias - dr.d * (m + j);
                            if (kLo <= kHi) {
                                best.H.x = j == c.n[0] ? max(best.H.x, (int)(mx & 0xffffu) + off) : best.H.x;
                                best.H.y = j == c.n[1] ? max(best.H.y, (int)(mx >> 16) + off) : best.H.y;
                            }
                        }
                    }
                }
            }
            if constexpr (LOC)
                dcol += QD;
            // The last block's stores are never read as values inside the band.
#pragma unroll
            for (int u = 0; u < QD; ++u) {
                rb[((s0 + u) & cm) * 64] = outv[u];
                rq[u] = nx[u];
            }
            if constexpr (LR)
                pg.publish(s0 + QD - 1);
        };
        int s0 = jA, g = gS;
        // The group's residue bytes; the next group's dwords are loaded
        // before a group and shifted after it, so the loop head waits for
        // nothing (a wait there would also cover the last group's stores).
        uint32_t curA = __builtin_amdgcn_alignbyte(a1, a0, shA);
        uint32_t curB = __builtin_amdgcn_alignbyte(b1, b0, shB);
        // Consecutive groups share a dword: one new dword per pair and group,
        // loaded two groups before its use.
        uint32_t a2 = ra.words[min(wA + gS + 2, ra.lastW)], b2w = rbs.words[min(wB + gS + 2, rbs.lastW)];
        auto next = [&](auto edge) {
            const uint32_t a3 = ra.words[min(wA + g + 3, ra.lastW)];
            const uint32_t b3 = rbs.words[min(wB + g + 3, rbs.lastW)];
            group(edge, s0, curA, curB);
            curA = __builtin_amdgcn_alignbyte(a2, a1, shA);
            curB = __builtin_amdgcn_alignbyte(b2w, b1, shB);
            a1 = a2;
            b1 = b2w;
            a2 = a3;
            b2w = b3;
            s0 += QD;
            ++g;
        };
        // The lower boundary's columns, the plain columns, the upper
        // boundary's columns (one loop: a single copy of the boundary form).
        while (s0 <= jEnd) {
            next(std::true_type{});
            if (s0 - jS >= R)
                while (s0 <= jEnd && s0 - jS + QD - 1 < W1)
                    next(std::false_type{});
        }
        if constexpr (LOC)
            best.b2 = sub(b2, (uint32_t)dcol * (uint32_t)dr.d * 0x10001u);
        if constexpr (LR) {
            pg.publish(0xffff);
        } else {
            // The next block reads this block's row-buffer entries from the
            // same lane: order the stores before those loads.
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        }
    }

    // Work item: `first` .. first + (count & 0xffff) of `order`, all of length
    // m = count >> 16; nblocks = (m + R) / R; maxN the largest n.
    __device__ __forceinline__ static bool wellFormed(const FwdArgs &a, const WorkItem &w)
    {
        const int pairs = w.count & 0xffff, m = (int)((uint32_t)w.count >> 16);
        return !(pairs < 1 || pairs > 128 || w.maxN < 1 || a.bandCols < 1 || (a.bandCols & (a.bandCols - 1)) != 0 ||
                 a.bandCols > a.rowCols || (a.bandCols < bandRowCols(w.maxN) && a.bandCols < a.bandUp - a.bandLo + R + 10) ||
                 m < 1 || w.nblocks != (m + R) / R);
    }

    __device__ __forceinline__ static void run(const FwdArgs &a)
    {
        __shared__ uint32_t sProf[16];
        __shared__ int16_t sT[33 * 33];
        // t = s - o, and the second half of a diagonal step's drift (global);
        // the rows' padding code: 0, or what keeps a free first row at H = 0
        // (-gapOpen; DNA: a byte, the caller takes the table form above 255).
        const int tAdd = LOC ? 0 : a.drift.d;
        const int padScore = !LOC && (a.mode & SQMI_FREE_TOP) ? a.drift.cost + a.drift.d : 0;
        if constexpr (DNA) {
            if (threadIdx.x < 16) {
                uint32_t w = a.dnaProfile[threadIdx.x];
                if ((int)threadIdx.x >= 8 && (int)threadIdx.x - 8 < a.alpha)
                    w += (uint32_t)tAdd * (0x01010101u >> (32 - 8 * min(a.alpha, 4)));
                sProf[threadIdx.x] = (int)threadIdx.x - 8 == a.alpha ? (uint32_t)padScore * 0x01010101u : w;
            }
        } else {
            const int TW = a.alpha + 1;
            for (int i = threadIdx.x; i < TW * TW; i += blockDim.x)
                sT[i] = i / TW == a.alpha ? (int16_t)0 : i % TW == a.alpha ? (int16_t)padScore : (int16_t)(a.tTable[i] + tAdd);
        }
        __syncthreads();

        const int lane = threadIdx.x & 63;
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const int waves = (int)(blockDim.x >> 6);
        __shared__ uint32_t sProg[kBandWaves], sItem;
        __shared__ int2 sBest[LR ? kBandWaves * 64 : 1];
        uint2 *rb;
        if constexpr (LR) {
            extern __shared__ uint2 sRing[];
            rb = sRing + lane;
        } else {
            rb = reinterpret_cast<uint2 *>(a.rowbuf) + ((size_t)blockIdx.x * waves + wave) * (size_t)a.rowCols * 64 + lane;
        }
        for (;;) {
            int it;
            if constexpr (LR) {
                if (threadIdx.x == 0)
                    sItem = atomicAdd(a.queue, 1u);
                if (threadIdx.x < kBandWaves)
                    sProg[threadIdx.x] = 0;
                __syncthreads();
                it = (int)sItem;
                __syncthreads();   // read by every wave before it is set again
            } else {
                // Branch-free fetch: every lane takes part (lane 0 adds 1).
                it = (int)atomicAdd(a.queue, lane == 0 ? 1u : 0u);
            }
            it = __builtin_amdgcn_readfirstlane(it);
            if (it >= a.nItems)
                break;
            const WorkItem w = a.items[it];
            if (!wellFormed(a, w))
                continue;
            const int pairs = w.count & 0xffff, m = (int)((uint32_t)w.count >> 16);
            Couple c;
            int minN = INT32_MAX;
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int sidx = 2 * lane + x;
                const int pid = sidx < pairs ? a.order[w.first + sidx] : -1;
                int64_t ho = 0, vo = 0;
                int n = 0;
                if (pid >= 0) {
                    ho = a.hOff[pid];
                    vo = a.vOff[pid];
                    n = (int)(a.hOff[pid + 1] - ho);
                    minN = min(minN, n);
                }
                c.h[x] = a.hRes + ho;
                c.v[x] = a.vRes + vo;
                c.n[x] = n;
                c.pid[x] = pid;
            }
            if constexpr (FREE) {
#pragma unroll
                for (int q = 1; q < 64; q <<= 1)
                    minN = min(minN, __shfl_xor(minN, q));
                minN = __builtin_amdgcn_readfirstlane(minN);
            }
            Best best{make_int2(INT32_MIN, INT32_MIN), (uint32_t)(a.drift.bias - a.drift.cost) * 0x10001u};
            const int p = w.nblocks * R - 1 - m;   // item row of row 0
            for (int b = LR ? wave : 0; b < w.nblocks; b += LR ? waves : 1) {
                Progress pg{};
                if constexpr (LR)
                    pg = Progress{sProg + (b + waves - 1) % waves, sProg + wave, (uint32_t)(b - 1) << 16, (uint32_t)b << 16, a.error};
                block(a, c, b * R - p, w.maxN, minN, b == 0, b == w.nblocks - 1, rb, sProf, sT, best, pg);
            }
            if constexpr (LOC)
                best.H = make_int2((int)(best.b2 & 0xffffu) + a.drift.cost - a.drift.bias,
                                   (int)(best.b2 >> 16) + a.drift.cost - a.drift.bias);
            if constexpr (LR) {
                sBest[wave * 64 + lane] = best.H;
                __syncthreads();
                if (wave != 0)
                    continue;
                for (int q = 1; q < waves; ++q) {
                    const int2 o = sBest[q * 64 + lane];
                    best.H = make_int2(max(best.H.x, o.x), max(best.H.y, o.y));
                }
            }
            if (c.pid[0] >= 0)
                a.scores[c.pid[0]] = best.H.x;
            if (c.pid[1] >= 0)
                a.scores[c.pid[1]] = best.H.y;
        }
    }
};

template <int R, bool DNA, int KIND, bool WIDE, bool LR>
__global__ __launch_bounds__(LR ? 64 * kBandWaves : 256) __attribute__((amdgpu_waves_per_eu(2))) void kBand16(FwdArgs a)
{
    Band16<R, DNA, KIND, WIDE, LR>::run(a);
}

}  // namespace
}  // namespace sqmi
