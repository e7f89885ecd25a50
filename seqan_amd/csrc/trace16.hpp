// trace16.hpp -- the packed int16 trace kernels (kTrace16): the forward pass
// with the trace bits of every cell, global under every AlignConfig and
// local, for gfx950.  Instantiated per DNA profile / substitution table by
// trace16.hip.
//
// The sweep is the score kernel's (score16.hpp): drifted values, LDS rings,
// strips; blocks of 256 rows, by 16 lanes of 16 rows each per pair couple, or
// by 64 lanes of 4 rows (a step takes a third of the time).  Per
// cell four decisions are recorded, which is what dp_formula_affine.h:62-126
// and _maxScore (dp_formula.h:165-201) record, ties resolved the same way:
//   E  E(i,j) opened a gap:    E(i,j-1) + e <  G(i,j-1)   (TraceBitMap_ HORIZONTAL_OPEN)
//   F  F(i,j) opened a gap:    F(i-1,j) + e <  G(i-1,j)   (VERTICAL_OPEN)
//   D  H(i,j) is not diagonal: D < max(E, F)              (not DIAGONAL)
//   X  E beats F:              F < E                      (MAX_FROM_HORIZONTAL_MATRIX)
// Drift keeps each comparison (both sides carry the same cell's drift; where
// extending costs more than reopening, e < o, E and F always count as opened,
// and the walk takes the bit as set).  Each is the sign of a saturating
// packed difference; two differences' signs become bytes with one v_perm_b32
// and go into the record with one v_bfi_b32.  Per packed row that is 14
// operations (wide: 15) against 17 in plain values.
//
// Per lane and column step one 16-byte record; bit kk of each byte is row kk
// (x, z: rows 0-7; y, w: rows 8-15) and the bytes are
//   x, y: E of pair A, E of pair B, F of pair A, F of pair B
//   z, w: D of pair A, D of pair B, X of pair A, X of pair B.
// Records of block b, step s of an item sit at trace[(traceOff[item] + b *
// steps + s) * 64 + lane]: one coalesced 1 KB store per wave and step.  With
// 64 lanes a record is one word, x | z << 4 (four rows), and a step 256 bytes.
//
// What bounds it: vector issue while there are items for every wave (65,536
// pairs of 1 kbp: 93% of the slots, 15.3 instructions per packed row with the
// lookup and the sweep's own; local 96%, 23); with few items, the sweep of the
// longest, which strips spread over the chip and 64 lanes per couple shorten
// (8,191 uneven pairs: 49%).  Measured: 65,536 pairs of 1 kbp, global, 17.4 ->
// 15.0 ms (34 GB of records at 2.4 TB/s beside it); 8,191 uneven pairs, free
// first and last row, 277 ms with one wave per item -> 8.6 (strips) -> 3.1 (64
// lanes); 8,192 protein pairs, local, 11.3 -> 2.9 ms.  The DNA kernels spill 38 to
// 247 registers of their four bodies' set-up at three waves per SIMD; the
// column loops read none back.
//
// Values are compared as signed halves.  WIDE: stored values are held less
// 32768, so that the whole 16-bit range is ordered and the differences
// saturate with the right sign.
//
// End cells (dp_scout.h:169-210, dp_scout_simd.h:427-440): every unit leaves
// its candidates (TraceEnd) and the walk takes the first strict maximum in
// the reference's order.
#pragma once

#include "score16.hpp"

namespace sqmi {
namespace {

constexpr int kTOutWords = 4 * kPeriod + 64 + kPeriod;
// Bottom rows with E beside G and F (the end cell's E and F).
__shared__ uint4 gOutE[kWaves * kTOutWords];

__device__ __forceinline__ uint32_t signBytes(s16x2 t0, s16x2 t1)
{
    // v_perm_b32 selectors 8..11 replicate bits 15, 31 (of the second
    // operand) and 47, 63 (of the first) into whole bytes: {sign(t0.x),
    // sign(t0.y), sign(t1.x), sign(t1.y)} as 0x00 / 0xFF.
    return __builtin_amdgcn_perm(asu(t1), asu(t0), 0x0B0A0908u);
}
__device__ __forceinline__ int half16(uint32_t w, int x) { return (int)(int16_t)(x ? w >> 16 : w); }

template <int G, bool DNA, uint32_t TRK, bool WIDE>
struct Trace16 {
    static constexpr bool LOC = (TRK & kTrackLocal) != 0;
    static constexpr int RB = kTraceRows / G, GROUPS = 64 / G, QD = kQD, P = kPeriod, RING = kRing<G>;
    // A lane's record of a step (file head).
    using Rec = std::conditional_t<G == 16, uint4, uint32_t>;

    __device__ __forceinline__ static uint32_t add(uint32_t a, uint32_t b) { return WIDE ? uadd2(a, b) : a + b; }
    __device__ __forceinline__ static uint32_t sub(uint32_t a, uint32_t b) { return WIDE ? usub2(a, b) : a - b; }
    __device__ __forceinline__ static uint32_t vmaxu(uint32_t a, uint32_t b) { return asu(vmax(as16(a), as16(b))); }
    __device__ __forceinline__ static uint32_t max3(uint32_t a, uint32_t b, uint32_t c)
    {
        return WIDE ? vmaxu(vmaxu(a, b), c) : max3Pos(a, b, c);
    }

    // Per lane: its best candidate cell (bottom row or, local, any cell) and
    // its best cell of column n, per pair; values in H.
    struct Cand {
        int v[2], i[2], j[2], e[2], f[2];
    };

    template <bool HEAD>
    __device__ __forceinline__ static void sweep(const TraceArgs &a, Couple c, int top, const bool last,
                                                 const bool strip, int Nw, const uint64_t *rowIn, uint64_t *rowOut,
                                                 const uint32_t *sProf, const char *sT, Rec *trBlock, Cand &cb,
                                                 Cand &cr, bool &stop)
    {
        // Opaque copies, as in the score kernel.
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        Drift dr = a.drift;
        dr.d = __builtin_amdgcn_readfirstlane(dr.d);
        dr.cost = __builtin_amdgcn_readfirstlane(dr.cost);
        dr.neg = __builtin_amdgcn_readfirstlane(dr.neg);
        dr.bias = __builtin_amdgcn_readfirstlane(dr.bias);
        Nw = __builtin_amdgcn_readfirstlane(Nw);
        top = __builtin_amdgcn_readfirstlane(top);
        if constexpr (WIDE) {
            dr.neg -= 32768;
            dr.bias -= 32768;
        }
        const int lane = tid & 63, l = lane % G, grp = lane / G;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const bool leftFree = (a.mode & SQMI_FREE_LEFT) != 0, topFree = (a.mode & SQMI_FREE_TOP) != 0;
        const int PAD = a.alpha, TW = a.alpha + 1;
        const int rowbase = top + l * RB;
        const uint32_t neg2 = asu(splat(dr.neg));
        uint32_t cost2 = (uint32_t)dr.cost * 0x10001u, d2 = (uint32_t)dr.d * 0x10001u;
        asm volatile("" : "+v"(cost2), "+v"(d2));

        uint32_t raw[2][RB];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int top1 = rowbase - c.p[x] - 1, lim = max(c.m[x] - 1, 0);
#pragma unroll
            for (int k = 0; k < RB; ++k)
                raw[x][k] = c.v[x][min(max(top1 + k, 0), lim)];
        }
        uint32_t selA[RB], selB[DNA ? 1 : RB], Gk[RB], Ek[RB], rowK[HEAD && !LOC ? RB : 1];
        const int border = leftFree ? dr.bias - dr.cost : dr.bias - 2 * dr.cost;
        const int slope = leftFree ? dr.d : 0;
#pragma unroll
        for (int k = 0; k < RB; ++k) {
            uint32_t sel[2];
            int g0[2], e0[2], fl[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int i = rowbase + k - c.p[x];
                const uint32_t cc = i >= 1 ? min(raw[x][k], (uint32_t)PAD) : (uint32_t)PAD;
                if constexpr (DNA)
                    sel[x] = cc < 4 ? cc + 4 * x : 0x0cu;
                else
                    sel[x] = cc * (4 * kTabCopies) + 4u * (uint32_t)(lane & (kTabCopies - 1));
                if constexpr (LOC) {
                    g0[x] = e0[x] = dr.neg;
                } else {
                    int g = border + slope * max(i, 0);
                    e0[x] = dr.neg;
                    if constexpr (HEAD) {
                        g = i == 0 ? dr.bias - dr.cost : g;
                        g = i < 0 ? dr.neg : g;
                        e0[x] = i == 0 && topFree ? dr.bias : dr.neg;
                        fl[x] = i == 0 && topFree ? dr.d : 0;
                    }
                    g0[x] = g;
                }
            }
            if constexpr (DNA) {
                selA[k] = sel[0] | (sel[1] << 16) | 0x0c000c00u;
            } else {
                selA[k] = sel[0] + 2;
                selB[k] = sel[1];
            }
            Gk[k] = asu(pack(g0[0], g0[1]));
            Ek[k] = asu(pack(e0[0], e0[1]));
            if constexpr (HEAD && !LOC)
                rowK[k] = (uint32_t)fl[0] | ((uint32_t)fl[1] << 16);
        }
        // H of a stored G, E, F at (i, j): less the drift and the bias.
        auto hOfG = [&](int g, int ij) { return g + dr.cost - dr.bias - dr.d * ij; };
        auto hOf = [&](int g, int ij) { return g - dr.bias - dr.d * ij; };

        constexpr int CPL = G == 16 ? 2 : 1;   // columns per lane of a refill (G = 64: lanes 0..31)
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
                const int j = colOf(s, q), x = (j + G - 1) & (RING - 1);
                uint4 w;
                w.x = prof(j >= 1 && j <= c.n[0] ? min((int)hr[0][q], PAD) : PAD);
                w.y = prof(j >= 1 && j <= c.n[1] ? min((int)hr[1][q], PAD) : PAD);
                w.z = w.w = neg2;
                if constexpr (!HEAD) {
                    w.z = (uint32_t)rv[q];
                    w.w = (uint32_t)(rv[q] >> 32);
                    if constexpr (WIDE) {   // words in memory are never 0 (stored values)
                        w.z ^= 0x80008000u;
                        w.w ^= 0x80008000u;
                    }
                }
                if constexpr (LOC) {
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

        uint4 *outBase = gOutE + wave * kTOutWords;
        uint4 *outLane = l == G - 1 ? outBase + grp * P : outBase + 4 * P + lane;
        auto rowWord = [&](uint32_t g, uint32_t f) -> uint64_t {
            const uint32_t flip = WIDE ? 0x80008000u : 0u;
            return ((uint64_t)(f ^ flip) << 32) | (g ^ flip);
        };
        auto flush = [&](int s1, int cnt) {
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < CPL; ++q) {
                const int idx = G == 16 ? 2 * l + q : l, j = s1 - cnt + idx - (G - 1);
                if (idx >= cnt || j < 1 || j > Nw)
                    continue;
                const uint4 w = outBase[grp * P + idx];
                if (!last) {
                    uint32_t g = w.x, f = w.y;
                    if constexpr (LOC) {
                        const uint32_t up = (uint32_t)((idx & (kRebase - 1)) + 1) * d2;
                        g = sub(g, up);
                        f = sub(f, up);
                    }
                    rowStore(rowOut + j, rowWord(g, f), strip);
                } else if constexpr (!LOC && (TRK & (kTrackBottom | kTrackEnd))) {
#pragma unroll
                    for (int x = 0; x < 2; ++x) {
                        // With a free last column, (m, n) is tracked there.
                        const bool in = (TRK & kTrackEnd) ? j == c.n[x] : (TRK & kTrackRight) ? j < c.n[x] : j <= c.n[x];
                        const int v = hOfG(half16(w.x, x), c.m[x] + j);
                        if (in && v > cb.v[x]) {
                            cb.v[x] = v;
                            cb.i[x] = c.m[x];
                            cb.j[x] = j;
                            cb.e[x] = hOf(half16(w.z, x), c.m[x] + j);
                            cb.f[x] = hOf(half16(w.y, x), c.m[x] + j);
                        }
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
        };

        uint32_t botG = Gk[RB - 1], botF = neg2, upGprev = neg2;
        uint32_t z2 = asu(splat(dr.bias));                              // local: the stored 0
        // Local: G of the lane's best cell so far (a whole item's earlier
        // blocks included), H >= 1.
        uint32_t best2 = asu(pack(dr.bias - dr.cost + max(LOC ? cb.v[0] : 0, 1),
                                  dr.bias - dr.cost + max(LOC ? cb.v[1] : 0, 1)));
        constexpr int DL = 4;
        uint32_t qa[DNA ? 1 : DL], qb[DNA ? 1 : DL];
        auto ldA = [&](uint32_t col, int k) -> uint32_t { return *reinterpret_cast<const uint16_t *>(sT + (col + selA[k])); };
        auto ldB = [&](uint32_t col, int k) -> uint32_t { return *reinterpret_cast<const uint32_t *>(sT + (col + selB[k])); };

        auto step = [&](auto chk, int s, int u, const uint4 &cur, const uint4 &nxt, uint4 *out) {
            constexpr bool CHK = decltype(chk)::value;
            const int j = s - l;
            const uint32_t upG = shiftIn<G>(botG, cur.z), upF = shiftIn<G>(botF, cur.w);
            uint32_t diagTop = upGprev;
            upGprev = upG;
            uint32_t botE = 0;
            if constexpr (LOC) {
                diagTop = add(diagTop, d2);
                best2 = add(best2, d2);
                if (CHK && j <= 1) {
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
                uint32_t accEF0 = 0, accEF1 = 0, accDX0 = 0, accDX1 = 0;
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
                        return WIDE ? uadd2(g, ta | tb) : g + ta + tb;
                    }
                };
                uint32_t D = dOf(diagTop, 0);
#pragma unroll
                for (int k = 0; k < RB; ++k) {
                    uint32_t Ex = Ek[k];
                    if constexpr (HEAD && !LOC)
                        Ex = add(Ex, rowK[k]);
                    const uint32_t ef = signBytes(subSat(as16(Ex), as16(Gk[k])), subSat(as16(uF), as16(uG)));
                    const uint32_t E = LOC ? max3(Ex, Gk[k], z2) : vmaxu(Ex, Gk[k]);
                    uint32_t F = vmaxu(uF, uG);
                    if (LOC && k > 0)
                        F = sub(F, d2);
                    Ek[k] = E;
                    const uint32_t H = max3(D, E, F);   // D < max(E, F) is D < H
                    const uint32_t dx = signBytes(subSat(as16(D), as16(H)), subSat(as16(F), as16(E)));
                    // Insert bit kk of every byte.  Written as v_bfi_b32
                    // statements so that each row's bits are taken while its
                    // values are live (left to itself the compiler defers all
                    // 16 rows to one OR tree and needs ~250 registers).
                    const uint32_t bit = 0x01010101u << (k & 7);
                    if (k < 8) {
                        asm volatile("v_bfi_b32 %0, %1, %2, %0" : "+v"(accEF0) : "s"(bit), "v"(ef));
                        asm volatile("v_bfi_b32 %0, %1, %2, %0" : "+v"(accDX0) : "s"(bit), "v"(dx));
                    } else {
                        asm volatile("v_bfi_b32 %0, %1, %2, %0" : "+v"(accEF1) : "s"(bit), "v"(ef));
                        asm volatile("v_bfi_b32 %0, %1, %2, %0" : "+v"(accDX1) : "s"(bit), "v"(dx));
                    }
                    if (k + 1 < RB)
                        D = dOf(Gk[k], k + 1);
                    Gk[k] = sub(H, cost2);
                    uG = Gk[k];
                    uF = F;
                    if constexpr (LOC)
                        m2 = k == 0 ? uG : vmaxu(m2, uG);
                }
                botG = uG;
                botF = uF;
                botE = Ek[RB - 1];
                if constexpr (LOC) {
                    // The first strict maximum over every cell in column
                    // order.  The column's maximum first; the rows are
                    // scanned only when it reaches the best so far (equal
                    // values count when they lie in an earlier column: a
                    // later block sweeps columns the earlier ones passed).
                    if (gtMask(as16(m2), as16(usub2(best2, 0x00010001u))) != 0) {
                        const uint32_t earlier = (j < cb.j[0] ? 0xffffu : 0u) | (j < cb.j[1] ? 0xffff0000u : 0u);
                        const uint32_t take = gtMask(as16(m2), as16(best2)) | (eqMask(as16(m2), as16(best2)) & earlier);
                        if (take != 0) {
                            uint32_t open = 0xffffffffu;   // halves whose first maximal row is still ahead
                            uint32_t rowK2 = 0, selE = 0, selF = 0;
                            uint32_t Fr = vmaxu(upF, upG);
#pragma unroll
                            for (int k = 0; k < RB; ++k) {
                                if (k > 0)
                                    Fr = sub(vmaxu(Fr, Gk[k - 1]), d2);
                                const uint32_t below = asu(subSat(as16(Gk[k]), as16(m2)) >> splat(15));
                                const uint32_t first = ~below & open;
                                open &= below;
                                rowK2 = bfi(first, (uint32_t)k * 0x10001u, rowK2);
                                selE = bfi(first, Ek[k], selE);
                                selF = bfi(first, Fr, selF);
                            }
                            best2 = bfi(take, m2, best2);
                            const int k1 = (s & (kRebase - 1)) + 1;   // the step's drift
#pragma unroll
                            for (int x = 0; x < 2; ++x)
                                if (take & (x ? 0xffff0000u : 0xffffu)) {
                                    cb.v[x] = hOfG(half16(m2, x), k1);
                                    cb.i[x] = rowbase + (int)((rowK2 >> (16 * x)) & 0xffffu) - c.p[x];
                                    cb.j[x] = j;
                                    cb.e[x] = hOf(half16(selE, x), k1);
                                    cb.f[x] = hOf(half16(selF, x), k1);
                                }
                        }
                    }
                }
                if constexpr (TRK & kTrackRight) {
                    // The lane's rows of column n in row order; F of each row
                    // again from the column above it.
                    if (j == c.n[0] || j == c.n[1]) {
                        uint32_t Fr = vmaxu(upF, upG);
#pragma unroll
                        for (int k = 0; k < RB; ++k) {
                            if (k > 0)
                                Fr = vmaxu(Fr, Gk[k - 1]);
#pragma unroll
                            for (int x = 0; x < 2; ++x) {
                                const int i = rowbase + k - c.p[x];
                                const int v = hOfG(half16(Gk[k], x), i + j);
                                if (j == c.n[x] && i >= 0 && v > cr.v[x]) {
                                    cr.v[x] = v;
                                    cr.i[x] = i;
                                    cr.j[x] = j;
                                    cr.e[x] = hOf(half16(Ek[k], x), i + j);
                                    cr.f[x] = hOf(half16(Fr, x), i + j);
                                }
                            }
                        }
                    }
                }
                if constexpr (G == 16)
                    trBlock[(size_t)s * 64] = make_uint4(accEF0, accEF1, accDX0, accDX1);
                else
                    trBlock[(size_t)s * 64] = accEF0 | accDX0 << 4;
            }
            out[u] = make_uint4(botG, botF, botE, 0);
        };

        const int steps = (Nw + G + QD - 1) / QD * QD;
        refillLoad(0);
        refillStore(0);
        // Column 0 of the bottom row: for the next block, or a tracked cell
        // (its E and F are minus infinity: it is never entered by a gap rule).
        const uint32_t g00 = LOC ? asu(splat(dr.bias - dr.cost)) : Gk[RB - 1];
        if (l == G - 1) {
            if (!last) {
                rowStore(rowOut, rowWord(g00, neg2), strip);
            } else if constexpr (!LOC && (TRK & kTrackBottom)) {
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const int v = hOfG(half16(g00, x), c.m[x]);
                    if (c.n[x] > 0 && v > cb.v[x]) {
                        cb.v[x] = v;
                        cb.i[x] = c.m[x];
                        cb.j[x] = 0;
                        cb.e[x] = cb.f[x] = INT32_MIN;
                    }
                }
            }
        }
        refillLoad(P);
        uint4 cur = ring[(G - 1 - l) & (RING - 1)];
        auto chunk = [&](auto chk, int s0) {
            if ((s0 & (P - 1)) == P - QD) {
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
            const uint4 *rr = ring + ((s0 + G - l) & (RING - 1));
            uint4 *out = outLane + (s0 & (P - 1));
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
        for (; s0 < min(LOC ? G + QD : G, steps); s0 += QD)
            chunk(std::true_type{}, s0);
        if constexpr (!DNA) {
#pragma unroll
            for (int k = 0; k < DL; ++k) {
                qa[k] = ldA(cur.x, k);
                qb[k] = ldB(cur.y, k);
            }
        }
        for (; s0 < steps; s0 += QD)
            chunk(std::false_type{}, s0);
        if (steps & (P - 1))
            flush(steps, steps & (P - 1));
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }

    // The lanes' candidates of a couple reduced to lane 0's: larger value,
    // then smaller column, then smaller row.
    __device__ __forceinline__ static void reduce(Cand &q)
    {
#pragma unroll
        for (int d = 1; d < G; d <<= 1)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int v = __shfl_xor(q.v[x], d, G), i = __shfl_xor(q.i[x], d, G), j = __shfl_xor(q.j[x], d, G);
                const int e = __shfl_xor(q.e[x], d, G), f = __shfl_xor(q.f[x], d, G);
                const bool t = v > q.v[x] || (v == q.v[x] && (j < q.j[x] || (j == q.j[x] && i < q.i[x])));
                q.v[x] = t ? v : q.v[x];
                q.i[x] = t ? i : q.i[x];
                q.j[x] = t ? j : q.j[x];
                q.e[x] = t ? e : q.e[x];
                q.f[x] = t ? f : q.f[x];
            }
    }

    __device__ __forceinline__ static void unit(const TraceArgs &a, const ScoreUnit &w, uint64_t *slotRow,
                                                const uint32_t *sProf, const char *sT, bool &stop)
    {
        const int lane = threadIdx.x & 63, l = lane % G, grp = lane / G;
        const int pairs = w.count, nb = w.nblocks, item = w.pad;
        const bool strip = w.block >= 0;
        const int stride = w.maxN + 1, steps = (w.maxN + G + QD - 1) / QD * QD;
        const int64_t rec0 = a.traceOff[item];
        // (A step of one couple on 64 lanes takes a quarter of one of four on 16.)
        constexpr int Q = G == 16 ? 1 : 4;
        if (pairs < 1 || pairs > 2 * GROUPS || w.maxN < 1 || nb < 1 || nb > (1 << 15) || w.block >= nb ||
            rec0 < 0 || Q * rec0 + (int64_t)nb * steps > Q * a.traceRecs ||
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
            c.p[x] = kTraceRows * nb - 1 - m;
        }
        Cand cb, cr;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            cb.v[x] = cr.v[x] = LOC ? 0 : INT32_MIN;
            cb.i[x] = cr.i[x] = cb.j[x] = cr.j[x] = 0x7fffffff;
            cb.e[x] = cr.e[x] = cb.f[x] = cr.f[x] = INT32_MIN;
        }
        Rec *tr = reinterpret_cast<Rec *>(a.trace + (size_t)rec0 * 64) + lane;
        const int b0 = strip ? w.block : 0, b1 = strip ? w.block + 1 : nb;
        for (int b = b0; b < b1; ++b) {
            const bool last = b == nb - 1;
            const uint64_t *in = strip ? a.strips + w.rowOff + ((int64_t)(b - 1) * GROUPS + grp) * stride
                                       : slotRow + (int64_t)grp * stride;
            uint64_t *out = strip ? a.strips + w.rowOff + ((int64_t)b * GROUPS + grp) * stride : slotRow + (int64_t)grp * stride;
            Rec *trBlock = tr + (size_t)b * steps * 64;
            if (b == 0)
                sweep<true>(a, c, 0, last, strip, w.maxN, in, out, sProf, sT, trBlock, cb, cr, stop);
            else
                sweep<false>(a, c, b * kTraceRows, last, strip, w.maxN, in, out, sProf, sT, trBlock, cb, cr, stop);
        }
        reduce(cb);
        if constexpr (TRK & kTrackRight)
            reduce(cr);
        if (l == 0) {
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                if (c.pid[x] < 0)
                    continue;
                // Candidates of strip b of the item's pairs, b-major.
                TraceEnd *t = a.ends + a.endOff[item] + (int64_t)b0 * pairs + (2 * grp + x);
                *t = TraceEnd{cb.v[x], cb.i[x], cb.j[x], cb.e[x], cb.f[x], cr.v[x], cr.i[x], cr.j[x], cr.e[x], cr.f[x]};
            }
        }
    }
};

template <bool DNA, uint32_t TRK>
__device__ __forceinline__ void traceRun(const TraceArgs &a)
{
    __shared__ uint32_t sProf[8];
    __shared__ __align__(16) char sT[DNA ? 16 : kTabLdsBytes];
    loadScores<DNA>(a, (TRK & kTrackLocal) ? 0 : a.drift.d, sProf, sT);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint64_t *slotRow = a.rowbuf + (size_t)(blockIdx.x * (blockDim.x >> 6) + wave) * a.slotWords;
    bool stop = false;
    for (;;) {
        int it = (int)atomicAdd(a.queue, lane == 0 ? 1u : 0u);   // branch-free, as in the score kernel
        it = __builtin_amdgcn_readfirstlane(it);
        if (it >= a.nUnits)
            break;
        const ScoreUnit w = uniformUnit(a.units[it]);
        if (w.shape & kUnit64) {
            if (w.shape & kUnitWide)
                Trace16<64, DNA, TRK, true>::unit(a, w, slotRow, sProf, sT, stop);
            else
                Trace16<64, DNA, TRK, false>::unit(a, w, slotRow, sProf, sT, stop);
        } else {
            if (w.shape & kUnitWide)
                Trace16<16, DNA, TRK, true>::unit(a, w, slotRow, sProf, sT, stop);
            else
                Trace16<16, DNA, TRK, false>::unit(a, w, slotRow, sProf, sT, stop);
        }
    }
}

template <bool DNA, uint32_t TRK>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DNA ? 3 : 2))) void kTrace16(TraceArgs a)
{
    traceRun<DNA, TRK>(a);
}

}  // namespace
}  // namespace sqmi
