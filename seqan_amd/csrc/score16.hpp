// score16.hpp -- the packed int16 score kernels (kScore16): exact affine-gap
// scores, global under every AlignConfig and local, for gfx950.
// Instantiated per DNA profile / substitution table and kind by score16.hip.
//
// Recurrence: SeqAn 2's Gotoh formula (include/seqan/align/
// dp_formula_affine.h:62-126), its borders (dp_formula_affine.h:244-330,
// dp_formula.h:289-309) and result cells (dp_meta_info.h:178-221,
// dp_scout.h:169-210).  Two pairs share every 32-bit register (the low and
// high 16-bit halves).  What bounds the kernel is the issue of vector
// instructions, so the values are held in a form that needs few of them:
//
// Global (drifted values, kernels.hpp): a gap extension adds nothing, every
// value is >= 0, and a cell is
//   E = max(E, G); F = max(F, G); H = max3(D, E, F); G = H - cost; D' = G + t
// i.e. five operations and one score lookup against eight and one in plain
// values.  max3 is v_pk_maximum3_f16 on the bit patterns (non-negative finite
// halves order like integers); sums and differences are 32-bit operations on
// both halves at once, which issue faster than packed 16-bit ones.  Measured
// on 1 M uneven DNA pairs, semi-global (6.8e11 cells): 65.5 ms against 91.8,
// 6.4 instructions per packed cell in the steady loop against 9.0 (6.7 over the
// whole launch), 92% of the issue slots (3.65e10 vector instructions of the
// waves at 4 cycles in 65.5 ms at 2.38 GHz).  (32-bit sums issue every 2.4 cycles among themselves but not beside packed ones.)
//
// Local: values are drifted by the step s of the sweep alone, stored = value
// + drift * (s mod kRebase + 1) + bias, and the registers are rebased every
// kRebase steps, so the range does not grow with the length.  (F of a lane's
// first row needs no subtraction: its neighbour's values are one step old.)  The floor H >= 0 rides in E's maximum (E >= z, z the stored 0):
//   E = max3(E, G, z); F = max(F, G) - drift; H = max3(D, E, F); G = H - cost
// and one maximum per two rows keeps the best cell: 6.5 operations and the
// lookup against 9.  262,144 protein pairs (Blosum62): 20.35 ms against 27.2, 91%
// of the issue slots, 9.8 instructions per packed cell.
//
// WIDE (values past kDriftNarrowMax, or scores t < 0): the same recurrences
// in packed 16-bit operations with two maxima for max3.
//
// Sweep.  A group of G lanes takes a pair couple; each lane owns RB
// consecutive rows of a block of G * RB rows and the group walks the columns
// as a skewed wavefront: at step s lane l computes column s - l and receives
// the bottom cell of lane l - 1 by a DPP move.  Rows are bottom-aligned: row m
// is the last row of the last block; block 0 is as tall as the item needs.
// The columns' profile words and the bottom row of the block above come from
// a per-group LDS ring (one 16-byte read per step), refilled every 32 steps
// from loads issued 32 steps earlier; the block's own bottom row goes to a
// small LDS buffer that is written out every 32 steps.  The step loop itself
// touches no global memory.
//
// Work units.  A unit is a whole item (all its row blocks, one after the
// other, on one wave) or one row block of an item (a strip): the blocks of a
// long item are swept by different waves at once, anywhere on the chip, each
// a few dozen columns behind the one above.  A strip's bottom row travels
// through global memory as 8-byte words that are stored and loaded with
// agent scope; the buffer starts zeroed and no stored word is 0, so a word is
// its own ready flag and no fence is needed.  Units are claimed from one
// counter in list order, and a strip only waits for the strip before it in
// the list, which an earlier claim handed to a running wave: the unfinished
// claimed unit with the lowest index always has its inputs, so every wait
// ends.  Waits are bounded all the same (about four seconds); past the bound
// the wave raises a flag in host memory and no wave waits any more.
#pragma once

#include <type_traits>

#include "kernels.hpp"
#include "packed16.hpp"
#include "seqan_amd.h"

namespace sqmi {
namespace {

// Lane l of every group of G lanes receives v from lane l-1; lane 0 of the
// group receives its own `first`.  One DPP move whose lanes without a source
// keep the old value: row_shr:1 for rows of 16 lanes, wave_shr:1 for 64.
template <int G>
__device__ __forceinline__ uint32_t shiftIn(uint32_t v, uint32_t first)
{
    static_assert(G == 16 || G == 64, "groups of 16 lanes or whole wavefronts");
    constexpr int ctrl = G == 16 ? 0x111 : 0x138;
    return (uint32_t)__builtin_amdgcn_update_dpp((int)first, (int)v, ctrl, 0xf, 0xf, false);
}

// Waves per workgroup, independent of each other: at most 4, or 8 where they
// share a table of 32 copies (score kernels).
#if defined(SQMI_SCORE_DNA) && !SQMI_SCORE_DNA
constexpr int kWaves = kScoreTabWaves, kTabCopies = 32;
#else
constexpr int kWaves = 4, kTabCopies = 16;
#endif
constexpr int kPeriod = 32;      // steps between refills of the ring and flushes of the bottom row
constexpr int kQD = 4;           // steps per chunk
constexpr int kRebase = 16;      // local: steps between rebases of the drift

// Ring entry of a column: profile words (DNA: t bytes for v = 0..3; table:
// byte offset of the column's words) of pairs A and B, and G and F of the row
// above the block.  Lane l reads entry s - l + G - 1 at step s.  The live
// columns span G - 1 back and kPeriod + 1 ahead: 64 entries for G = 16, 128
// for G = 64, then a copy of the first kQD so that a chunk reads from one
// base.
template <int G> constexpr int kRing = G == 16 ? 64 : 128;
constexpr int kRingWords = kWaves * 4 * (kRing<16> + kQD);
static_assert(4 * (kRing<16> + kQD) >= kRing<64> + kQD, "a wave's rings fit both group sizes");
__shared__ uint4 gRing[kRingWords];
// Bottom rows: per wave kPeriod entries per group (at most 4), then the
// entries the other lanes' writes go to (their values are not used).
constexpr int kOutWords = 4 * kPeriod + 64 + kPeriod;
__shared__ uint2 gOut[kWaves * kOutWords];

// Substitution table of the table kernels in LDS: word (h, v), copy c of
// kTabCopies, holds t << 16 (lane c mod kTabCopies reads its own copy).  Pair
// A reads the word's high half (t), pair B the word (t << 16).  With 32 copies
// the 32 lanes that read at once never meet in a bank; with 16 two lanes do
// whenever their words agree modulo 4.  The trace kernels have no room for 32
// beside their rings.  262,144 protein pairs, local: 21.0 -> 20.35 ms, 64 to 65,536 of them
// 1-4% faster.
constexpr int kTabLdsBytes = kTabMaxCodes * kTabMaxCodes * 4 * kTabCopies;

__device__ __forceinline__ uint64_t rowLoad(const uint64_t *p, bool strip)
{
    return strip ? __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                 : __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void rowStore(uint64_t *p, uint64_t v, bool strip)
{
    if (strip)
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// A refill's words of the strip above (columns j0, j0 + 1, ... of the lane):
// waits until they are there.  Ends: see the file's head; `stop` once a wait
// has run past its bound.
template <int C>
__device__ __forceinline__ void waitWords(uint64_t (&rv)[C], const uint64_t *rowIn, int Nw, int j0, uint32_t *error,
                                          bool &stop)
{
    int spins = 0;
    for (;;) {
        bool missing = false;
#pragma unroll
        for (int q = 0; q < C; ++q)
            missing |= (uint32_t)rv[q] == 0;
        if (stop || __ballot(missing) == 0)
            break;
        __builtin_amdgcn_s_sleep(8);
        if (++spins > (1 << 21)) {
            __hip_atomic_store(error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            stop = true;
        } else if ((spins & 1023) == 0) {
            stop = __hip_atomic_load(error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0;
        }
#pragma unroll
        for (int q = 0; q < C; ++q)
            if ((uint32_t)rv[q] == 0)
                rv[q] = rowLoad(rowIn + min(max(j0 + q, 0), Nw), true);
    }
}

// The unit's fields as wave-uniform values.
__device__ __forceinline__ ScoreUnit uniformUnit(ScoreUnit w)
{
    w.first = __builtin_amdgcn_readfirstlane(w.first);
    w.count = __builtin_amdgcn_readfirstlane(w.count);
    w.maxN = __builtin_amdgcn_readfirstlane(w.maxN);
    w.nblocks = __builtin_amdgcn_readfirstlane(w.nblocks);
    w.rows = __builtin_amdgcn_readfirstlane(w.rows);
    w.shape = __builtin_amdgcn_readfirstlane(w.shape);
    w.block = __builtin_amdgcn_readfirstlane(w.block);
    w.pad = __builtin_amdgcn_readfirstlane(w.pad);
    return w;
}

// The score tables in LDS: t = s - o + tAdd for real codes, 0 for the padding
// code (tAdd: the drift under drift in both directions, the diagonal step's
// second half; 0 local).
template <bool DNA, class Args>
__device__ __forceinline__ void loadScores(const Args &a, int tAdd, uint32_t *sProf, char *sT)
{
    if constexpr (DNA) {
        if (threadIdx.x < 5) {
            uint32_t w = a.dnaProfile[threadIdx.x];
            if ((int)threadIdx.x < a.alpha)
                w += (uint32_t)tAdd * (0x01010101u >> (32 - 8 * min(a.alpha, 4)));
            sProf[threadIdx.x] = w;
        }
    } else {
        // A word per thread, its copies from the lane's own on, so that the
        // lanes' stores spread over the banks.
        const int TW = a.alpha + 1;
        for (int w = threadIdx.x; w < TW * TW; w += blockDim.x) {
            const int h = w / TW, v = w % TW;
            const uint32_t t = (h == a.alpha || v == a.alpha) ? 0u : (uint32_t)(uint16_t)(a.tTable[w] + tAdd);
            for (int c = 0; c < kTabCopies; ++c)
                *reinterpret_cast<uint32_t *>(sT + 4 * (w * kTabCopies + (((int)threadIdx.x + c) & (kTabCopies - 1)))) = t << 16;
        }
    }
    __syncthreads();
}

// Per-lane state of one pair couple (lo = pair A, hi = pair B).
struct Couple {
    const uint8_t *h[2];
    const uint8_t *v[2];
    int n[2], m[2], p[2], pid[2];   // p: item row of the pair's row 0
};

template <int G, bool DNA, int KIND, bool WIDE>
struct Score16 {
    static constexpr bool LOC = KIND == kScoreLocal, RIGHT = KIND == kScoreRight;
    static constexpr int GROUPS = 64 / G, QD = kQD, P = kPeriod, RING = kRing<G>;

    // Sums, differences and maxima of both halves.  Narrow values stay below
    // 0x8000, so no carry or borrow crosses the halves.
    __device__ __forceinline__ static uint32_t add(uint32_t a, uint32_t b) { return WIDE ? uadd2(a, b) : a + b; }
    __device__ __forceinline__ static uint32_t sub(uint32_t a, uint32_t b) { return WIDE ? usub2(a, b) : a - b; }
    __device__ __forceinline__ static uint32_t max3(uint32_t a, uint32_t b, uint32_t c)
    {
        return WIDE ? umax2(umax2(a, b), c) : max3Pos(a, b, c);
    }

    // One block of rows from item row `top` (lane 0's first row): HEAD for
    // block 0.  last: the block holding row m.  rowIn / rowOut: bottom row of
    // the block above / of this block, by column.
    template <bool HEAD, int RB>
    __device__ __forceinline__ static void sweep(const ScoreArgs &a, Couple c, int top, const bool last,
                                                 const bool strip, int Nw, const uint64_t *rowIn, uint64_t *rowOut,
                                                 const uint32_t *sProf, const char *sT, int2 &bestH, bool &stop)
    {
        // Opaque copies: what a block derives from the lane, the couple and
        // the scoring is made anew in each block, instead of being hoisted
        // out of all of them and spilled.
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        Drift dr = a.drift;
        dr.d = __builtin_amdgcn_readfirstlane(dr.d);
        dr.cost = __builtin_amdgcn_readfirstlane(dr.cost);
        dr.neg = __builtin_amdgcn_readfirstlane(dr.neg);
        dr.bias = __builtin_amdgcn_readfirstlane(dr.bias);
        Nw = __builtin_amdgcn_readfirstlane(Nw);
        top = __builtin_amdgcn_readfirstlane(top);
        const int lane = tid & 63, l = lane % G, grp = lane / G;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const bool leftFree = (a.mode & SQMI_FREE_LEFT) != 0, topFree = (a.mode & SQMI_FREE_TOP) != 0;
        const bool bottomFree = (a.mode & SQMI_FREE_BOTTOM) != 0;
        const int PAD = a.alpha, TW = a.alpha + 1;
        const int rowbase = top + l * RB;
        const uint32_t neg2 = (uint32_t)dr.neg * 0x10001u;
        // In vector registers: 32-bit operations with a scalar operand issue
        // at half the rate.
        uint32_t cost2 = (uint32_t)dr.cost * 0x10001u, d2 = (uint32_t)dr.d * 0x10001u;
        asm volatile("" : "+v"(cost2), "+v"(d2));

        // Rows: residue selectors, column 0.  Global: G(i, 0) and E = -inf;
        // row 0 under a free top takes E(0, j) = H(0, j) = E(0, j - 1) +
        // drift (rowK).  Local: set at the lane's first column.
        // All residue loads first (clamped into the pair), so that a block
        // waits once for them.
        uint32_t raw[2][RB];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int top1 = rowbase - c.p[x] - 1, lim = max(c.m[x] - 1, 0);
#pragma unroll
            for (int k = 0; k < RB; ++k)
                raw[x][k] = c.v[x][min(max(top1 + k, 0), lim)];
        }
        uint32_t selA[RB], selB[DNA ? 1 : RB], Gk[RB], Ek[RB], rowK[HEAD && !LOC ? RB : 1];
        const int border = leftFree ? dr.bias - dr.cost : dr.bias - 2 * dr.cost;   // G(i, 0), i >= 1, less
        const int slope = leftFree ? dr.d : 0;                                      // slope * i
#pragma unroll
        for (int k = 0; k < RB; ++k) {
            uint32_t sel[2], g0[2], e0[2], fl[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int i = rowbase + k - c.p[x];
                const uint32_t cc = i >= 1 ? min(raw[x][k], (uint32_t)PAD) : (uint32_t)PAD;
                if constexpr (DNA)
                    sel[x] = cc < 4 ? cc + 4 * x : 0x0cu;
                else
                    sel[x] = cc * (4 * kTabCopies) + 4u * (uint32_t)(lane & (kTabCopies - 1));
                if constexpr (LOC) {
                    g0[x] = e0[x] = (uint32_t)dr.neg;
                } else {
                    int g = border + slope * max(i, 0);
                    if constexpr (HEAD) {
                        g = i == 0 ? dr.bias - dr.cost : g;
                        g = i < 0 ? dr.neg : g;
                        e0[x] = (uint32_t)(i == 0 && topFree ? dr.bias : dr.neg);
                        fl[x] = (uint32_t)(i == 0 && topFree ? dr.d : 0);
                    } else {
                        e0[x] = (uint32_t)dr.neg;
                    }
                    g0[x] = (uint32_t)g & 0xffffu;
                }
            }
            if constexpr (DNA) {
                selA[k] = sel[0] | (sel[1] << 16) | 0x0c000c00u;
            } else {
                selA[k] = sel[0] + 2;   // the word's high half
                selB[k] = sel[1];
            }
            Gk[k] = g0[0] | (g0[1] << 16);
            Ek[k] = e0[0] | (e0[1] << 16);
            if constexpr (HEAD && !LOC)
                rowK[k] = fl[0] | (fl[1] << 16);
        }
        const int base[2] = {dr.cost - dr.bias - dr.d * c.m[0], dr.cost - dr.bias - dr.d * c.m[1]};
        // Residues and row entries of a refill: columns j0 (and j0 + 1 for
        // G = 16) of lane l, loaded a period before they go to the ring.
        constexpr int CPL = G == 16 ? 2 : 1;   // columns per lane (G = 64: lanes 0..31)
        uint4 *ring = gRing + wave * 4 * (kRing<16> + QD) + (G == 16 ? grp * (kRing<16> + QD) : 0);
        uint32_t hr[2][CPL];
        uint64_t rv[CPL];
        auto colOf = [&](int s, int q) { return G == 16 ? s + 2 * l + q : s + (l & (P - 1)); };
        auto refillLoad = [&](int s) {
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
                const int j = colOf(s, q);
#pragma unroll
                for (int x = 0; x < 2; ++x)
                    hr[x][q] = c.h[x][min(max(j, 1), max(c.n[x], 1)) - 1];
                if constexpr (!HEAD)
                    rv[q] = rowLoad(rowIn + min(max(j, 0), Nw), strip);
            }
        };
        auto prof = [&](int code) -> uint32_t {
            if constexpr (DNA)
                return sProf[code];
            else
                return (uint32_t)(code * TW * 4 * kTabCopies);
        };
        auto refillStore = [&](int s) {
            if constexpr (!HEAD) {
                if (strip)
                    waitWords(rv, rowIn, Nw, colOf(s, 0), a.error, stop);
            }
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
                const int j = colOf(s, q);
                const int x = (j + G - 1) & (RING - 1);
                uint4 w;
                w.x = prof(j >= 1 && j <= c.n[0] ? min((int)hr[0][q], PAD) : PAD);
                w.y = prof(j >= 1 && j <= c.n[1] ? min((int)hr[1][q], PAD) : PAD);
                w.z = w.w = neg2;
                if constexpr (!HEAD) {
                    w.z = (uint32_t)rv[q];
                    w.w = (uint32_t)(rv[q] >> 32);
                }
                if constexpr (LOC) {
                    // Entry j meets lane 0 at step j, as a value of the step
                    // before (HEAD: G of a row of zeros).
                    const uint32_t up = (uint32_t)(j & (kRebase - 1)) * d2;
                    w.z = add(w.z, up);
                    w.w = add(w.w, up);
                }
                if (G == 16 || l < P) {
                    ring[x] = w;
                    if (x < QD)
                        ring[x + RING] = w;
                }
            }
            __builtin_amdgcn_wave_barrier();
        };

        // Bottom row: the group's last lane writes entry s mod P at step s,
        // the other lanes elsewhere.
        uint2 *outBase = gOut + wave * kOutWords;
        uint2 *outLane = l == G - 1 ? outBase + grp * P : outBase + 4 * P + lane;
        auto flush = [&](int s1, int cnt) {   // the entries of steps s1 - cnt .. s1 - 1
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
                const int idx = G == 16 ? 2 * l + q : l;
                if (idx >= cnt)
                    continue;
                const int j = s1 - cnt + idx - (G - 1);
                uint2 w = outBase[grp * P + idx];
                if (j < 1 || j > Nw)
                    continue;
                if (!last) {
                    if constexpr (LOC) {
                        const uint32_t up = (uint32_t)((idx & (kRebase - 1)) + 1) * d2;
                        w.x = sub(w.x, up);
                        w.y = sub(w.y, up);
                    }
                    rowStore(rowOut + j, ((uint64_t)w.y << 32) | w.x, strip);
                } else if constexpr (!LOC) {
                    if (bottomFree ? j <= c.n[0] : (!RIGHT && j == c.n[0]))
                        bestH.x = max(bestH.x, (int)(w.x & 0xffffu) + base[0] - dr.d * j);
                    if (bottomFree ? j <= c.n[1] : (!RIGHT && j == c.n[1]))
                        bestH.y = max(bestH.y, (int)(w.x >> 16) + base[1] - dr.d * j);
                }
            }
            __builtin_amdgcn_wave_barrier();
        };

        uint32_t botG = Gk[RB - 1], botF = neg2, upGprev = neg2;
        uint32_t z2 = (uint32_t)dr.bias * 0x10001u;     // local: the stored 0 of the current step
        uint32_t best2 = (uint32_t)dr.neg * 0x10001u;   // local: the best G so far, at the current drift

        // Table lookups run DL rows ahead, through DL slots (t of pair A, t
        // << 16 of pair B); the last rows of a step read the next column's.
        constexpr int DL = RB % 4 == 0 ? 4 : RB % 2 == 0 ? 2 : 1;
        uint32_t qa[DNA ? 1 : DL], qb[DNA ? 1 : DL];
        auto ldA = [&](uint32_t col, int k) -> uint32_t { return *reinterpret_cast<const uint16_t *>(sT + (col + selA[k])); };
        auto ldB = [&](uint32_t col, int k) -> uint32_t { return *reinterpret_cast<const uint32_t *>(sT + (col + selB[k])); };

        // One column of the lane's rows.  CHK: the lane may still be left of
        // its first column (the first G steps).  Columns past n are computed
        // like the others: their scores are 0, which adds nothing to any
        // value, and no result is taken from them.
        auto step = [&](auto chk, int s, int u, const uint4 &cur, const uint4 &nxt, uint2 *out) {
            constexpr bool CHK = decltype(chk)::value;
            const int j = s - l;
            const uint32_t upG = shiftIn<G>(botG, cur.z), upF = shiftIn<G>(botF, cur.w);
            uint32_t diagTop = upGprev;
            upGprev = upG;
            if constexpr (LOC) {
                // Neighbour values are one step old, diagonal ones two.
                diagTop = add(diagTop, d2);
                best2 = add(best2, d2);
                if (CHK && j <= 1) {
                    // Column 0 at the drift of the step before.
                    const uint32_t g = sub(z2, cost2);
#pragma unroll
                    for (int k = 0; k < RB; ++k) {
                        Gk[k] = g;
                        Ek[k] = z2;
                    }
                    diagTop = g;
                    botG = add(g, d2);
                    botF = g;
                }
                z2 = add(z2, d2);
            }
            if (!CHK || j >= 1) {
                uint32_t uG = upG, uF = upF, m2 = 0;
                auto dOf = [&](uint32_t g, int k) -> uint32_t {
                    if constexpr (DNA) {
                        return add(g, __builtin_amdgcn_perm(cur.y, cur.x, selA[k]));
                    } else {
                        uint32_t ta, tb;
                        if constexpr (!CHK) {
                            ta = qa[k % DL];
                            tb = qb[k % DL];
                            const int kn = k + DL;
                            qa[k % DL] = kn < RB ? ldA(cur.x, kn) : ldA(nxt.x, kn - RB);
                            qb[k % DL] = kn < RB ? ldB(cur.y, kn) : ldB(nxt.y, kn - RB);
                        } else {
                            ta = ldA(cur.x, k);
                            tb = ldB(cur.y, k);
                        }
                        return WIDE ? uadd2(g, ta | tb) : g + ta + tb;   // narrow: t >= 0, one v_add3_u32
                    }
                };
                uint32_t D = dOf(diagTop, 0);
#pragma unroll
                for (int k = 0; k < RB; ++k) {
                    uint32_t E, F;
                    if constexpr (LOC) {
                        E = max3(Ek[k], Gk[k], z2);
                        F = umax2(uF, uG);
                        if (k > 0)
                            F = sub(F, d2);
                    } else {
                        E = Ek[k];
                        if constexpr (HEAD)
                            E = add(E, rowK[k]);
                        E = umax2(E, Gk[k]);
                        F = umax2(uF, uG);
                    }
                    Ek[k] = E;
                    const uint32_t H = max3(D, E, F);
                    if (k + 1 < RB)
                        D = dOf(Gk[k], k + 1);
                    Gk[k] = sub(H, cost2);
                    uG = Gk[k];
                    uF = F;
                    if constexpr (LOC) {
                        if (RB == 1)
                            m2 = uG;
                        else if (k % 2 == 1)
                            m2 = k == 1 ? umax2(Gk[0], uG) : max3(m2, Gk[k - 1], uG);
                        else if (k == RB - 1)
                            m2 = umax2(m2, uG);
                    }
                }
                botG = uG;
                botF = uF;
                if constexpr (LOC)
                    best2 = umax2(best2, m2);
                if constexpr (RIGHT) {
                    // The maximum of the lane's rows in column n, per half.
                    // Going down the rows the running maximum gains drift
                    // per row, so that it stays comparable with the next
                    // row's stored value; rows above row 0 are left out.
                    if (j == c.n[0] || j == c.n[1]) {
                        const int iTop[2] = {rowbase - c.p[0], rowbase - c.p[1]};
                        uint32_t mx = Gk[0];
#pragma unroll
                        for (int k = 1; k < RB; ++k) {
                            mx = uadd2(mx, d2);
                            if constexpr (HEAD)
                                mx &= ~((iTop[0] + k - 1 < 0 ? 0xffffu : 0u) | (iTop[1] + k - 1 < 0 ? 0xffff0000u : 0u));
                            mx = umax2(mx, Gk[k]);
                        }
                        if (j == c.n[0] && iTop[0] + RB > 0)
                            bestH.x = max(bestH.x, (int)(mx & 0xffffu) + dr.cost - dr.bias - dr.d * (iTop[0] + RB - 1 + j));
                        if (j == c.n[1] && iTop[1] + RB > 0)
                            bestH.y = max(bestH.y, (int)(mx >> 16) + dr.cost - dr.bias - dr.d * (iTop[1] + RB - 1 + j));
                    }
                }
            }
            out[u] = make_uint2(botG, botF);
        };

        const int steps = (Nw + G + QD - 1) / QD * QD;   // the last lane reaches column Nw at step Nw + G - 1
        refillLoad(0);
        refillStore(0);
        // Column 0 of the bottom row: for the next block, or a tracked cell.
        // A whole item's blocks share one buffer: the entry is written once
        // the block above's has reached the ring.
        // (Local: stored values carry no drift, G(i, 0) = bias - cost.)
        const uint32_t g00 = LOC ? (uint32_t)(dr.bias - dr.cost) * 0x10001u : Gk[RB - 1];
        if (l == G - 1) {
            if (!last) {
                rowStore(rowOut, ((uint64_t)neg2 << 32) | g00, strip);
            } else if (!LOC && bottomFree) {
                bestH.x = max(bestH.x, (int)(g00 & 0xffffu) + base[0]);
                bestH.y = max(bestH.y, (int)(g00 >> 16) + base[1]);
            }
        }
        refillLoad(P);
        uint4 cur = ring[(G - 1 - l) & (RING - 1)];
        auto chunk = [&](auto chk, int s0) {
            if ((s0 & (P - 1)) == P - QD) {
                // The ring for the next P steps (read from the next step on),
                // and the loads of the refill after it.
                refillStore(s0 + QD);
                refillLoad(s0 + QD + P);
            }
            if constexpr (LOC) {
                if ((s0 & (kRebase - 1)) == 0 && s0 > 0) {
                    const uint32_t r = d2 * kRebase;
#pragma unroll
                    for (int k = 0; k < RB; ++k) {
                        Gk[k] = sub(Gk[k], r);
                        Ek[k] = sub(Ek[k], r);
                    }
                    botG = sub(botG, r);
                    botF = sub(botF, r);
                    upGprev = sub(upGprev, r);
                    z2 = sub(z2, r);
                    best2 = sub(best2, r);
                }
            }
            const uint4 *rr = ring + ((s0 + G - l) & (RING - 1));   // rr[u]: the entry of step s0 + u + 1
            uint2 *out = outLane + (s0 & (P - 1));
#pragma unroll
            for (int u = 0; u < QD; ++u) {
                const uint4 nxt = rr[u];
                step(chk, s0 + u, u, cur, nxt, out);
                cur = nxt;
            }
            if ((s0 & (P - 1)) == P - QD)
                flush(s0 + QD, P);
        };
        int s0 = 0;
        // (The last lane is at column 1 at step G.)
        for (; s0 < min(LOC ? G + QD : G, steps); s0 += QD)
            chunk(std::true_type{}, s0);
        if constexpr (!DNA) {
#pragma unroll
            for (int k = 0; k < DL; ++k) {
                qa[k] = ldA(cur.x, k);   // the first steady step's first rows
                qb[k] = ldB(cur.y, k);
            }
        }
        for (; s0 < steps; s0 += QD)
            chunk(std::false_type{}, s0);
        if (steps & (P - 1))
            flush(steps, steps & (P - 1));
        if constexpr (LOC) {
            const int off = dr.cost - dr.bias - dr.d * (((steps - 1) & (kRebase - 1)) + 1);
            bestH.x = max(bestH.x, (int)(best2 & 0xffffu) + off);
            bestH.y = max(bestH.y, (int)(best2 >> 16) + off);
        }
        // Make this block's row entries visible to the wave's next block.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }

    // One unit (see the file's head).  slotRow: the wave's own row buffer
    // (whole items); strips use a.strips at the unit's offset.
    __device__ __forceinline__ static void unit(const ScoreArgs &a, const ScoreUnit &w, uint64_t *slotRow,
                                                const uint32_t *sProf, const char *sT, bool &stop)
    {
        const int lane = threadIdx.x & 63, l = lane % G, grp = lane / G;
        const int R = w.rows & 0xff, RH = (w.rows >> 8) & 0xff;
        const int pairs = w.count, nb = w.nblocks;
        const bool strip = w.block >= 0;
        const int stride = w.maxN + 1;   // row-buffer columns 0..maxN per group
        // A malformed descriptor is skipped rather than allowed to run past
        // a buffer or loop without bound.
        if (pairs < 1 || pairs > 2 * GROUPS || w.maxN < 1 || nb < 1 || nb > (1 << 15) || w.block >= nb ||
            (strip ? w.rowOff < 0 || w.rowOff + (int64_t)nb * GROUPS * stride > a.stripWords
                   : (int64_t)GROUPS * stride > a.slotWords))
            return;
        Couple c;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int sidx = 2 * grp + x;
            const int pid = sidx < pairs ? a.order[w.first + sidx] : -1;
            int64_t ho = 0, vo = 0;
            int n = 0, m = 0;
            if (pid >= 0) {
                ho = a.hOff[pid];
                vo = a.vOff[pid];
                n = (int)(a.hOff[pid + 1] - ho);
                m = (int)(a.vOff[pid + 1] - vo);
            }
            c.h[x] = a.hRes + ho;
            c.v[x] = a.vRes + vo;
            c.n[x] = n;
            c.m[x] = m;
            c.pid[x] = pid;
            c.p[x] = G * (RH + (nb - 1) * R) - 1 - m;
        }
        int2 bestH = make_int2(INT32_MIN, INT32_MIN);
        const int b0 = strip ? w.block : 0, b1 = strip ? w.block + 1 : nb;
        for (int b = b0; b < b1; ++b) {
            const bool last = b == nb - 1;
            const uint64_t *in = strip ? a.strips + w.rowOff + ((int64_t)(b - 1) * GROUPS + grp) * stride
                                       : slotRow + (int64_t)grp * stride;
            uint64_t *out = strip ? a.strips + w.rowOff + ((int64_t)b * GROUPS + grp) * stride
                                  : slotRow + (int64_t)grp * stride;
            const int top = b == 0 ? 0 : G * (RH + (b - 1) * R);
#define SQMI_SWEEP(HEAD, RB)                                                                                    \
    case RB:                                                                                                    \
        sweep<HEAD, RB>(a, c, top, last, strip, w.maxN, in, out, sProf, sT, bestH, stop);                       \
        break;
            if (b == 0) {
                if constexpr (G == 64) {
                    switch (RH) {
                        SQMI_SWEEP(true, 1)
                        SQMI_SWEEP(true, 2)
                        SQMI_SWEEP(true, 3)
                        SQMI_SWEEP(true, 4)
                        SQMI_SWEEP(true, 6)
                        SQMI_SWEEP(true, 8)
                        SQMI_SWEEP(true, 12)
                        SQMI_SWEEP(true, 16)
                        default: break;
                    }
                } else {
                    switch (RH) {
                        SQMI_SWEEP(true, 4)
                        SQMI_SWEEP(true, 8)
                        SQMI_SWEEP(true, 12)
                        SQMI_SWEEP(true, 16)
                        default: break;
                    }
                }
            } else {
                if constexpr (G == 64) {
                    switch (R) {
                        SQMI_SWEEP(false, 4)
                        SQMI_SWEEP(false, 8)
                        SQMI_SWEEP(false, 16)
                        default: break;
                    }
                } else {
                    switch (R) {
                        SQMI_SWEEP(false, 8)
                        SQMI_SWEEP(false, 16)
                        default: break;
                    }
                }
            }
#undef SQMI_SWEEP
        }
        // Strips of a mode that tracks cells of every block meet in the
        // scores array, which starts at INT32_MIN for their pairs.
        const bool merge = strip && (LOC || RIGHT);
        if (strip && !merge && w.block != nb - 1)
            return;
#pragma unroll
        for (int d = 1; d < G; d <<= 1) {
            bestH.x = max(bestH.x, __shfl_xor(bestH.x, d, G));
            bestH.y = max(bestH.y, __shfl_xor(bestH.y, d, G));
        }
        if (l == 0) {
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int best = x ? bestH.y : bestH.x;
                if (c.pid[x] < 0)
                    continue;
                if (merge)
                    atomicMax(a.scores + c.pid[x], best);
                else
                    a.scores[c.pid[x]] = best;
            }
        }
    }
};

template <bool DNA, int KIND>
__device__ __forceinline__ void scoreRun(const ScoreArgs &a)
{
    __shared__ uint32_t sProf[8];
    __shared__ __align__(16) char sT[DNA ? 16 : kTabLdsBytes];
    loadScores<DNA>(a, KIND == kScoreLocal ? 0 : a.drift.d, sProf, sT);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint64_t *slotRow = a.rowbuf + (size_t)(blockIdx.x * (blockDim.x >> 6) + wave) * a.slotWords;
    bool stop = false;
    for (;;) {
        // Every lane takes part in the atomic (lane 0 adds 1, the others 0)
        // and the wave takes lane 0's old value: a branch on lane == 0 here
        // could be merged with the lane-0 store at a unit's end into
        // divergent paths around the loop's back edge.
        int it = (int)atomicAdd(a.queue, lane == 0 ? 1u : 0u);
        it = __builtin_amdgcn_readfirstlane(it);
        if (it >= a.nUnits)
            break;
        const ScoreUnit w = uniformUnit(a.slim ? a.slim[it].unit() : a.units[it]);
        if (w.shape & kUnit64) {
            if (w.shape & kUnitWide)
                Score16<64, DNA, KIND, true>::unit(a, w, slotRow, sProf, sT, stop);
            else
                Score16<64, DNA, KIND, false>::unit(a, w, slotRow, sProf, sT, stop);
        } else {
            if (w.shape & kUnitWide)
                Score16<16, DNA, KIND, true>::unit(a, w, slotRow, sProf, sT, stop);
            else
                Score16<16, DNA, KIND, false>::unit(a, w, slotRow, sProf, sT, stop);
        }
    }
}

// Three waves per SIMD (168 registers) with the DNA profile, two (256) with
// the table, whose row offsets and scores read ahead would spill at three.
template <bool DNA, int KIND>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(DNA ? 3 : 2))) void kScore16(ScoreArgs a)
{
    scoreRun<DNA, KIND>(a);
}

}  // namespace
}  // namespace sqmi
