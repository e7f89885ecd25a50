// long16.hip -- packed int16 kernels for long DNA pairs, global alignment:
// the forward sweep in strips (kLong16), the traceback's recomputation of
// trace records from checkpoints (kLong16Trace) and the walk (kLong16Walk).
//
// Recurrence, borders and trace decisions are those of the score and trace
// kernels (score16.hpp, trace16.hpp), in their drifted values: two pairs (a
// couple) share every register, a gap extension adds nothing and three maxima
// are one instruction.  What is different:
//
// Strips.  A wave sweeps 64 R rows of a couple, R per lane, over all columns.
// The strips of a couple are claimed top-down by any waves; a strip's bottom
// row goes through memory in words that are their own ready flags, so strip
// b + 1 runs about 100 columns behind strip b.  Units are claimed strip by
// strip over all couples: the strip above a claimed one is always claimed
// earlier, by a wave that runs, so every wait ends (and is bounded besides).
//
// Range.  Drifted values never fall by more than the cost of a gap along a
// row or a column, and grow by at most A = sMax + 2 drift per column or row,
// so the cells a wave holds at one step differ by about 64 (R + 1) A at most,
// however long the pair.  Each half of a wave keeps a base that is raised
// (and taken off every register) once the wave's top row has grown by
// kLongSlackV over its target, so that all values stay within (0,
// kDriftNarrowMax].  Bottom rows carry absolute values modulo 2^16: a word
// holds G + base and, as G + cost - F >= 0 of at most 15 bits, F; the 16th
// bit of each half is the ready flag.  The strip below takes off its own base.
//
// Checkpoints.  Every kLongT steps a wave stores its whole state (R rows of G
// and E, F of the last row, the diagonal input, the bases): 2 R + 4 words a
// lane, coalesced, in place of borders of tiles.  A step is a skewed column,
// so a tile of the traceback is the strip between two such states, and it is
// swept by the code that made them.
//
// Traceback.  A round recomputes a window of kWinChunks chunks of kLongT steps
// by `winStrips` strips around each pair's walk position, all at once, with
// four trace bits per cell; a wave takes two neighbouring chunks of one pair in
// its register halves.  Then a wave per pair walks: the lanes read the bits
// of the next 64 cells of the diagonal (or the gap), so a run of equal moves
// costs one memory wait.
//
// What bounds it: vector issue (6.6 instructions per packed cell, 80% of the
// slots on 64 pairs, whose last round of strips leaves SIMDs idle) once the
// strips fill the SIMDs, the sweep of one strip and the start of the ones below
// before.  64 pairs of 100 kbp (6.4e11 cells): forward 270 -> 67 ms against one
// launch per tile anti-diagonal with plain values, 8 rows per lane (16: 77, of
// which a fourth round of 64 strips on 1,024 SIMDs takes 16; 4: 76); records 6
// ms and walks 6 ms of 82 rounds, 43 before (one thread per pair walked);
// scores and counts 315 -> 80 ms.
#include <algorithm>

#include "score16.hpp"

namespace sqmi {
namespace {

__device__ __forceinline__ uint32_t usubSat2(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2, a),
                                                                      __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ int half(uint32_t w, int x) { return (int)(x ? w >> 16 : w & 0xffffu); }
// Half x of a in the low half, half x of b in the high one.
__device__ __forceinline__ uint32_t halves(uint32_t a, uint32_t b, int x)
{
    return x ? (a >> 16) | (b & 0xffff0000u) : (a & 0xffffu) | (b << 16);
}
__device__ __forceinline__ uint32_t signBytes2(uint32_t t0, uint32_t t1)
{
    return __builtin_amdgcn_perm(t1, t0, 0x0B0A0908u);   // trace16.hpp, signBytes
}

constexpr uint32_t kReady = 0x80008000u;

// A workgroup fills a CU: kRanks waves per SIMD.
constexpr int kRanks = 3, kLongWaves = 4 * kRanks;
constexpr int kLongRing = kRing<64> + kQD;
__shared__ uint4 gLongRing[kLongWaves * kLongRing];
__shared__ uint2 gLongOut[kLongWaves * kOutWords];

// Residue selectors of a lane's R rows and their column 0 (both halves).
template <int R>
struct Rows {
    uint32_t sel[R], G[R];
};
template <int R>
__device__ __forceinline__ void loadRows(Rows<R> &r, const uint8_t *const (&v)[2], const int (&m)[2], const int (&p)[2],
                                         int rowbase, const Drift &dr)
{
    uint32_t raw[2][R];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int k = 0; k < R; ++k)
            raw[x][k] = v[x][min(max(rowbase + k - p[x] - 1, 0), max(m[x] - 1, 0))];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        uint32_t sel[2], g[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int i = rowbase + k - p[x];
            const uint32_t c = i >= 1 ? min(raw[x][k], 4u) : 4u;
            sel[x] = c < 4 ? c + 4 * x : 0x0cu;
            g[x] = (uint32_t)(i < 0 ? dr.neg : i == 0 ? dr.bias - dr.cost : dr.bias - 2 * dr.cost);
        }
        r.sel[k] = sel[0] | (sel[1] << 16) | 0x0c000c00u;
        r.G[k] = g[0] | (g[1] << 16);
    }
}

__device__ __forceinline__ Drift uniformDrift(const Drift &d)
{
    return Drift{__builtin_amdgcn_readfirstlane(d.d), __builtin_amdgcn_readfirstlane(d.cost),
                 __builtin_amdgcn_readfirstlane(d.neg), __builtin_amdgcn_readfirstlane(d.bias)};
}

// G of the row above a strip (pair row i) in column 0.
__device__ __forceinline__ uint32_t borderG(int i, const Drift &dr)
{
    return (uint32_t)(i < 0 ? dr.neg : i == 0 ? dr.bias - dr.cost : dr.bias - 2 * dr.cost);
}

template <int R>
__device__ __forceinline__ void strip(const LongArgs &a, const LongCouple &cp, int b, const uint32_t *sProf, bool &stop)
{
    constexpr int G = 64, QD = kQD, P = kPeriod, RING = kRing<64>;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // as in the score kernel
    const Drift dr = uniformDrift(a.drift);
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int Nw = cp.maxN;
    const bool last = b == cp.nb - 1;
    const int top = b * 64 * R, rowbase = top + lane * R;
    const uint8_t *h[2], *v[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const int pid = max(cp.pid[x], 0);
        h[x] = a.hRes + a.hOff[pid];
        v[x] = a.vRes + a.vOff[pid];
    }
    uint32_t cost2 = (uint32_t)dr.cost * 0x10001u;
    asm volatile("" : "+v"(cost2));
    const uint32_t neg2 = (uint32_t)dr.neg * 0x10001u;
    uint32_t sel[R], Gk[R], Ek[R];
    {
        Rows<R> r;
        loadRows<R>(r, v, cp.m, cp.p, rowbase, dr);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            sel[k] = r.sel[k];
            Gk[k] = r.G[k];
            Ek[k] = neg2;
        }
    }
    // Row above: 0xffff in the halves where it is a row of the pair.
    const uint32_t above = (top - 1 - cp.p[0] >= 0 ? 0xffffu : 0u) | (top - 1 - cp.p[1] >= 0 ? 0xffff0000u : 0u);
    const uint32_t aboveG0 = borderG(top - 1 - cp.p[0], dr) | (borderG(top - 1 - cp.p[1], dr) << 16);
    const uint64_t *rowIn = a.rows + cp.rows + (int64_t)(b - 1) * (Nw + 1);   // b > 0 only
    uint64_t *rowOut = a.rows + cp.rows + (int64_t)b * (Nw + 1);              // not the last strip's

    int base[2] = {0, 0};
    auto base16 = [&]() -> uint32_t { return ((uint32_t)base[0] & 0xffffu) | ((uint32_t)base[1] << 16); };

    uint4 *ring = gLongRing + wave * kLongRing;
    uint32_t hr[2];
    uint64_t rv = 0;
    auto refillLoad = [&](int s) {
        const int j = s + (lane & (P - 1));
#pragma unroll
        for (int x = 0; x < 2; ++x)
            hr[x] = h[x][min(max(j, 1), max(cp.n[x], 1)) - 1];
        if (b > 0)
            rv = rowLoad(rowIn + min(max(j, 1), Nw), true);
    };
    auto refillStore = [&](int s) {
        const int j = s + (lane & (P - 1));
        uint4 w;
        w.x = sProf[j >= 1 && j <= cp.n[0] ? min((int)hr[0], 4) : 4];
        w.y = sProf[j >= 1 && j <= cp.n[1] ? min((int)hr[1], 4) : 4];
        w.z = w.w = neg2;
        if (b > 0) {
            for (int spins = 0; !stop;) {
                const bool missing = (uint32_t)(rv >> 32) == 0;
                if (__ballot(missing) == 0)
                    break;
                __builtin_amdgcn_s_sleep(8);
                if (++spins > (1 << 21)) {
                    __hip_atomic_store(a.error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    stop = true;
                } else if ((spins & 1023) == 0) {
                    stop = __hip_atomic_load(a.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0;
                }
                if (missing)
                    rv = rowLoad(rowIn + min(max(j, 1), Nw), true);
            }
            const uint32_t g = usub2((uint32_t)rv, base16());
            const uint32_t f = usubSat2(uadd2(g, cost2), (uint32_t)(rv >> 32) & ~kReady);
            w.z = bfi(above, g, neg2);
            w.w = bfi(above, f, neg2);
        }
        if (j < 1) {
            w.z = b > 0 ? aboveG0 : neg2;
            w.w = neg2;
        }
        const int x = (j + G - 1) & (RING - 1);
        if (lane < P) {
            ring[x] = w;
            if (x < QD)
                ring[x + RING] = w;
        }
        __builtin_amdgcn_wave_barrier();
    };

    uint2 *outBase = gLongOut + wave * kOutWords;
    uint2 *outLane = lane == G - 1 ? outBase : outBase + 4 * P + lane;
    auto flush = [&](int s1, int cnt) {   // the entries of steps s1 - cnt .. s1 - 1
        __builtin_amdgcn_wave_barrier();
        const int j = s1 - cnt + lane - (G - 1);
        if (lane < cnt && j >= 1 && j <= Nw && !last) {
            const uint2 w = outBase[lane];
            const uint32_t g = uadd2(w.x, base16()), f = usub2(uadd2(w.x, cost2), w.y) | kReady;
            rowStore(rowOut + j, ((uint64_t)f << 32) | g, true);
        }
        __builtin_amdgcn_wave_barrier();
    };

    uint32_t botG = Gk[R - 1], botF = neg2, upGprev = neg2;
    int endStep[2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
        endStep[x] = last && cp.pid[x] >= 0 ? cp.n[x] + G - 1 : -1;

    // CHK: lanes may still be left of column 1; END: the last strip, whose
    // last lane meets the pairs' end cells.
    auto step = [&](auto chk, auto end, int s, int u, const uint4 &cur, uint2 *out) {
        constexpr bool CHK = decltype(chk)::value, END = decltype(end)::value;
        const uint32_t upG = shiftIn<G>(botG, cur.z), upF = shiftIn<G>(botF, cur.w);
        const uint32_t diagTop = upGprev;
        upGprev = upG;
        if (!CHK || s >= lane + 1) {
            uint32_t uG = upG, uF = upF;
            uint32_t D = diagTop + __builtin_amdgcn_perm(cur.y, cur.x, sel[0]);
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const uint32_t E = umax2(Ek[k], Gk[k]), F = umax2(uF, uG);
                Ek[k] = E;
                const uint32_t H = max3Pos(D, E, F);
                if (k + 1 < R)
                    D = Gk[k] + __builtin_amdgcn_perm(cur.y, cur.x, sel[k + 1]);
                Gk[k] = H - cost2;
                uG = Gk[k];
                uF = F;
            }
            botG = uG;
            botF = uF;
        }
        out[u] = make_uint2(botG, botF);
        if (END && (s == endStep[0] || s == endStep[1])) {   // cell (m, n) of a pair: the last lane's last row
            if (lane == G - 1) {
#pragma unroll
                for (int x = 0; x < 2; ++x)
                    if (s == endStep[x]) {
                        const int off = base[x] - dr.bias - dr.d * (cp.m[x] + cp.n[x]);
                        a.scores[cp.pid[x]] = half(botG, x) + dr.cost + off;
                        a.endEF[2 * (int64_t)cp.pid[x]] = half(Ek[R - 1], x) + off;
                        a.endEF[2 * (int64_t)cp.pid[x] + 1] = half(botF, x) + off;
                    }
            }
        }
    };

    const int steps = longSteps(Nw);
    uint4 *state = a.state ? reinterpret_cast<uint4 *>(a.state + cp.state + (int64_t)b * cp.chunks * longStateWords(R) * 64) + lane
                           : nullptr;
    refillLoad(0);
    refillStore(0);
    refillLoad(P);
    uint4 cur = ring[(G - 1 - lane) & (RING - 1)];
    uint32_t pend = 0;   // what the next period's start takes off every register
    auto chunk = [&](auto chk, auto end, int s0) {
        if ((s0 & (P - 1)) == 0) {
            if (pend) {
#pragma unroll
                for (int k = 0; k < R; ++k) {
                    Gk[k] -= pend;
                    Ek[k] -= pend;
                }
                botG -= pend;
                botF -= pend;
                upGprev -= pend;
                pend = 0;
            }
            if ((s0 & (kLongT - 1)) == 0 && state) {
                uint4 *st = state + (int64_t)(s0 / kLongT) * (longStateWords(R) / 4) * 64;
#pragma unroll
                for (int k = 0; k < R; k += 4) {
                    st[(k / 4) * 64] = make_uint4(Gk[k], Gk[k + 1], Gk[k + 2], Gk[k + 3]);
                    st[((R + k) / 4) * 64] = make_uint4(Ek[k], Ek[k + 1], Ek[k + 2], Ek[k + 3]);
                }
                st[(2 * R / 4) * 64] = make_uint4(botF, upGprev, (uint32_t)base[0], (uint32_t)base[1]);
            }
        }
        if ((s0 & (P - 1)) == P - QD) {
            // The ring for the next P steps, at the base they will have, and
            // the loads of the refill after it.
            const int b0 = base[0], b1 = base[1];
            if (s0 >= G) {
                const uint32_t g = __builtin_amdgcn_readfirstlane(Gk[0]);
                const int r0 = half(g, 0) - a.target, r1 = half(g, 1) - a.target;
                const int t0 = r0 >= kLongSlackV ? r0 : 0, t1 = r1 >= kLongSlackV ? r1 : 0;
                pend = (uint32_t)t0 | ((uint32_t)t1 << 16);
                base[0] += t0;
                base[1] += t1;
            }
            refillStore(s0 + QD);
            base[0] = b0;
            base[1] = b1;
            refillLoad(s0 + QD + P);
        }
        const uint4 *rr = ring + ((s0 + G - lane) & (RING - 1));   // rr[u]: the entry of step s0 + u + 1
        uint2 *out = outLane + (s0 & (P - 1));
#pragma unroll
        for (int u = 0; u < QD; ++u) {
            const uint4 nxt = rr[u];
            step(chk, end, s0 + u, u, cur, out);
            cur = nxt;
        }
        if ((s0 & (P - 1)) == P - QD) {
            flush(s0 + QD, P);
            base[0] += (int)(pend & 0xffffu);
            base[1] += (int)(pend >> 16);
        }
    };
    int s0 = 0;
    for (; s0 < min(G, steps); s0 += QD)
        chunk(std::true_type{}, std::false_type{}, s0);   // (n + G - 1 >= G: no end cell yet)
    if (last)
        for (; s0 < steps; s0 += QD)
            chunk(std::false_type{}, std::true_type{}, s0);
    else
        for (; s0 < steps; s0 += QD)
            chunk(std::false_type{}, std::false_type{}, s0);
    if (steps & (P - 1))
        flush(steps, steps & (P - 1));
}

// One workgroup per CU.  A chain of strips moves at the pace of its slowest
// wave, so the waves of a SIMD must not be neighbours in the chains, some
// SIMDs holding more of its head than others: the first units go to one wave
// of each SIMD, the next ones to the second, and the earlier a unit, the higher
// its wave's priority.  The head third of the strips then runs at full speed
// everywhere, the others in the slots it leaves.  (64 pairs of 100 kbp, R =
// 16, three waves per SIMD: 110-119 ms in workgroups of four waves that claim
// as they come.)
template <int R>
__global__ __launch_bounds__(64 * kLongWaves) __attribute__((amdgpu_waves_per_eu(kRanks))) void kLong16(LongArgs a)
{
    __shared__ uint32_t sProf[8];
    loadScores<true>(a, a.drift.d, sProf, nullptr);
    const int lane = threadIdx.x & 63, rank = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8));
    const int perRank = 4 * gridDim.x;
    // (Only the order of the first claims: the wait is short and bounded.)
    for (int spins = 0; spins < 256; ++spins) {
        const int claimed = (int)__hip_atomic_load(a.queue, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (claimed >= min(rank * perRank, a.nUnits))
            break;
        __builtin_amdgcn_s_sleep(8);
    }
    bool stop = false;
    for (;;) {
        int it = (int)atomicAdd(a.queue, lane == 0 ? 1u : 0u);   // branch-free, as in the score kernel
        it = __builtin_amdgcn_readfirstlane(it);
        if (it >= a.nUnits)
            break;
        const int order = it / perRank;
        if (order == 0)
            __builtin_amdgcn_s_setprio(3);
        else if (order == 1)
            __builtin_amdgcn_s_setprio(2);
        else if (order == 2)
            __builtin_amdgcn_s_setprio(1);
        else
            __builtin_amdgcn_s_setprio(0);
        const int2 u = a.units[it];
        const int c = __builtin_amdgcn_readfirstlane(u.x), b = __builtin_amdgcn_readfirstlane(u.y);
        const LongCouple cp = a.couples[c];
        if (b >= cp.nb || cp.maxN < 1)
            continue;
        strip<R>(a, cp, b, sProf, stop);
    }
}

// The walk's state of a pair (couple 2 c + x).
enum { LW_I = 0, LW_J, LW_MODE, LW_PREV, LW_OPENS, LW_EXTS, LW_NOPS, LW_DONE };

// The window of a pair whose walk stands at (i, j): strips b0 - winStrips + 1
// .. b0, chunks c0 - kWinChunks + 1 .. c0.
struct Window {
    int b0, c0;
};
template <int R>
__device__ __forceinline__ Window windowOf(int p, int i, int j)
{
    return Window{(p + i) / (64 * R), (j + 63) / kLongT};
}

template <int R>
struct alignas(longRecBytes(R)) LongRec {   // trace bits of a lane's rows: E and F opened, not diagonal and E beats F (bytes: trace16.hpp)
    uint32_t w[R == 16 ? 4 : 2];
};

// Two chunks (c in the low half, c - 1 in the high one) of strip b of one
// pair, from their checkpoints.
template <int R>
__device__ __forceinline__ void traceChunks(const LongArgs &a, const LongCouple &cp, int x, int b, int c,
                                            const uint32_t *sProf, uint4 *ring, LongRec<R> *rec)
{
    constexpr int G = 64, P = kPeriod, RING = kRing<64>;
    const int lane = threadIdx.x & 63, Nw = cp.maxN;
    const Drift dr = uniformDrift(a.drift);
    const int pid = x ? cp.pid[1] : cp.pid[0], n = x ? cp.n[1] : cp.n[0], m = x ? cp.m[1] : cp.m[0];
    const int p = x ? cp.p[1] : cp.p[0];
    const uint8_t *h = a.hRes + a.hOff[pid], *v = a.vRes + a.vOff[pid];
    const int top = b * 64 * R;
    uint32_t cost2 = (uint32_t)dr.cost * 0x10001u;
    asm volatile("" : "+v"(cost2));
    const uint32_t neg2 = (uint32_t)dr.neg * 0x10001u;
    uint32_t sel[R], Gk[R], Ek[R], botF, upGprev, base16;
    {
        const uint8_t *const vv[2] = {v, v};
        const int m2[2] = {m, m}, p2[2] = {p, p};
        Rows<R> r;
        loadRows<R>(r, vv, m2, p2, top + lane * R, dr);
        const int64_t st0 = cp.state + (int64_t)b * cp.chunks * longStateWords(R) * 64;
        const uint4 *s0 = reinterpret_cast<const uint4 *>(a.state + st0 + (int64_t)min(c, cp.chunks - 1) * longStateWords(R) * 64) + lane;
        const uint4 *s1 = reinterpret_cast<const uint4 *>(a.state + st0 + (int64_t)max(c - 1, 0) * longStateWords(R) * 64) + lane;
#pragma unroll
        for (int k = 0; k < R; k += 4) {
            const uint4 g0 = s0[(k / 4) * 64], g1 = s1[(k / 4) * 64], e0 = s0[((R + k) / 4) * 64], e1 = s1[((R + k) / 4) * 64];
            Gk[k] = halves(g0.x, g1.x, x);
            Gk[k + 1] = halves(g0.y, g1.y, x);
            Gk[k + 2] = halves(g0.z, g1.z, x);
            Gk[k + 3] = halves(g0.w, g1.w, x);
            Ek[k] = halves(e0.x, e1.x, x);
            Ek[k + 1] = halves(e0.y, e1.y, x);
            Ek[k + 2] = halves(e0.z, e1.z, x);
            Ek[k + 3] = halves(e0.w, e1.w, x);
        }
        const uint4 t0 = s0[(2 * R / 4) * 64], t1 = s1[(2 * R / 4) * 64];
        botF = halves(t0.x, t1.x, x);
        upGprev = halves(t0.y, t1.y, x);
        base16 = ((x ? t0.w : t0.z) & 0xffffu) | ((x ? t1.w : t1.z) << 16);
#pragma unroll
        for (int k = 0; k < R; ++k)
            sel[k] = r.sel[k];
    }
    const int col0[2] = {c * kLongT, (c - 1) * kLongT};   // lane 0's column at local step 0
    const int iAbove = top - 1 - p;
    const uint64_t *rowIn = a.rows + cp.rows + (int64_t)(b - 1) * (Nw + 1);
    uint32_t hr[2];
    uint64_t rv[2] = {0, 0};
    auto refillLoad = [&](int s) {
        const int jj = s + (lane & (P - 1));
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            hr[y] = h[min(max(col0[y] + jj, 1), max(n, 1)) - 1];
            if (iAbove >= 0)
                rv[y] = rowIn[min(max(col0[y] + jj, 1), Nw)];
        }
    };
    auto refillStore = [&](int s) {
        const int jj = s + (lane & (P - 1));
        uint4 w;
        const int j0 = col0[0] + jj, j1 = col0[1] + jj;
        w.x = sProf[j0 >= 1 && j0 <= n ? min((int)hr[0], 4) : 4];
        w.y = sProf[j1 >= 1 && j1 <= n ? min((int)hr[1], 4) : 4];
        w.z = w.w = neg2;
        if (iAbove >= 0) {
            const uint32_t g = usub2(halves((uint32_t)rv[0], (uint32_t)rv[1], x), base16);
            const uint32_t f = usubSat2(uadd2(g, cost2), halves((uint32_t)(rv[0] >> 32), (uint32_t)(rv[1] >> 32), x) & ~kReady);
            // Column 0: the border, and no vertical gap.
            const uint32_t in = (j0 >= 1 ? 0xffffu : 0u) | (j1 >= 1 ? 0xffff0000u : 0u);
            w.z = bfi(in, g, borderG(iAbove, dr) * 0x10001u);
            w.w = bfi(in, f, neg2);
        }
        if (lane < P)
            ring[(jj + G - 1) & (RING - 1)] = w;
        __builtin_amdgcn_wave_barrier();
    };
    // The G - 1 columns before the chunk's first (read by the later lanes).
    for (int s = -2 * P; s <= 0; s += P) {
        refillLoad(s);
        refillStore(s);
    }
    refillLoad(P);
    uint32_t botG = Gk[R - 1];
    auto step = [&](auto chk, int s, const uint4 &cur) {
        constexpr bool CHK = decltype(chk)::value;
        const uint32_t upG = shiftIn<G>(botG, cur.z), upF = shiftIn<G>(botF, cur.w);
        const uint32_t diagTop = upGprev;
        upGprev = upG;
        uint32_t upd = 0xffffffffu;   // halves at column 1 or later
        if constexpr (CHK)
            upd = (col0[0] + s - lane >= 1 ? 0xffffu : 0u) | (col0[1] + s - lane >= 1 ? 0xffff0000u : 0u);
        uint32_t uG = upG, uF = upF;
        uint32_t accEF[2] = {0, 0}, accDX[2] = {0, 0};
        uint32_t D = diagTop + __builtin_amdgcn_perm(cur.y, cur.x, sel[0]);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t Gl = Gk[k], Ex = Ek[k];
            const uint32_t ef = signBytes2(asu(subSat(as16(Ex), as16(Gl))), asu(subSat(as16(uF), as16(uG))));
            const uint32_t E = umax2(Ex, Gl), F = umax2(uF, uG);
            const uint32_t H = max3Pos(D, E, F);
            const uint32_t dx = signBytes2(asu(subSat(as16(D), as16(H))), asu(subSat(as16(F), as16(E))));
            const uint32_t bit = 0x01010101u << (k & 7);
            asm volatile("v_bfi_b32 %0, %1, %2, %0" : "+v"(accEF[k >> 3]) : "s"(bit), "v"(ef));
            asm volatile("v_bfi_b32 %0, %1, %2, %0" : "+v"(accDX[k >> 3]) : "s"(bit), "v"(dx));
            if (k + 1 < R)
                D = Gl + __builtin_amdgcn_perm(cur.y, cur.x, sel[k + 1]);
            const uint32_t Gn = H - cost2;
            Ek[k] = CHK ? bfi(upd, E, Ex) : E;
            Gk[k] = CHK ? bfi(upd, Gn, Gl) : Gn;
            uG = Gn;
            uF = F;
        }
        botG = CHK ? bfi(upd, uG, botG) : uG;
        botF = CHK ? bfi(upd, uF, botF) : uF;
        LongRec<R> q;
        if constexpr (R == 16) {
            q.w[0] = accEF[0];
            q.w[1] = accEF[1];
            q.w[2] = accDX[0];
            q.w[3] = accDX[1];
        } else {
            q.w[0] = accEF[0];
            q.w[1] = accDX[0];
        }
        rec[(int64_t)s * 64 + lane] = q;
    };
    for (int s0 = 0; s0 < kLongT; s0 += P) {
        // The ring holds this period's entries; the next period's go in at
        // its end (entries of the last 2 P columns stay).
        for (int s = s0; s < s0 + P; ++s) {
            const uint4 cur = ring[(s + G - 1 - lane) & (RING - 1)];
            if (c <= 1 && s < G)
                step(std::true_type{}, s, cur);
            else
                step(std::false_type{}, s, cur);
        }
        __builtin_amdgcn_wave_barrier();
        refillStore(s0 + P);
        refillLoad(s0 + 2 * P);
    }
}

__shared__ uint4 gTraceRing[4 * kLongRing];

// Wave q of a pair's window: strip b0 - q / kWinCouples, chunks c0 - 2 (q mod
// kWinCouples) and the one before.  Workgroups of a pair have ids equal to its
// slot mod 8, as its walk's, so that both run on one XCD and share its L2.
constexpr int longWinBlocks(int R) { return (longWinStrips(R) * kWinCouples + 3) / 4; }
template <int R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(R == 16 ? 2 : 3))) void kLong16Trace(LongArgs a)
{
    __shared__ uint32_t sProf[8];
    loadScores<true>(a, a.drift.d, sProf, nullptr);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int per = longWinStrips(R) * kWinCouples;   // waves per pair
    const int g = blockIdx.x / 8;
    const int slot = g / longWinBlocks(R) * 8 + blockIdx.x % 8, q = g % longWinBlocks(R) * 4 + wave;
    if (slot >= 2 * a.nCouples || q >= per)
        return;
    const int x = slot & 1;
    const LongCouple cp = a.couples[slot >> 1];
    if ((x ? cp.pid[1] : cp.pid[0]) < 0)
        return;
    const int32_t *ws = a.walk + (int64_t)slot * kLongWalkInts;
    const int i = __builtin_amdgcn_readfirstlane(ws[LW_I]), j = __builtin_amdgcn_readfirstlane(ws[LW_J]);
    if (__builtin_amdgcn_readfirstlane(ws[LW_DONE]))
        return;
    const Window win = windowOf<R>(x ? cp.p[1] : cp.p[0], i, j);
    const int b = win.b0 - q / kWinCouples, c = win.c0 - 2 * (q % kWinCouples);
    if (b < 0 || c < 0)
        return;
    LongRec<R> *rec = reinterpret_cast<LongRec<R> *>(a.trace) + ((int64_t)slot * per + q) * kLongT * 64;
    traceChunks<R>(a, cp, x, b, c, sProf, gTraceRing + wave * kLongRing, rec);
}

__global__ void kLong16WalkInit(LongArgs a)
{
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= 2 * a.nCouples)
        return;
    const LongCouple cp = a.couples[slot >> 1];
    const int x = slot & 1, pid = cp.pid[x];
    int32_t *ws = a.walk + (int64_t)slot * kLongWalkInts;
    ws[LW_DONE] = pid < 0;
    if (pid < 0)
        return;
    const int score = a.scores[pid], endE = a.endEF[2 * (int64_t)pid], endF = a.endEF[2 * (int64_t)pid + 1];
    ws[LW_I] = cp.m[x];
    ws[LW_J] = cp.n[x];
    // End cell: F, then E, win ties (dp_algorithm_impl.h:1190-1207,
    // PreferGapsAtEnd_ dp_traceback_impl.h:115-122); the linear-gap walk
    // (gap open == gap extend) takes the cell's own direction.
    ws[LW_MODE] = a.linear ? 0 : endF == score ? 1 : endE == score ? 2 : 0;
    ws[LW_PREV] = ws[LW_OPENS] = ws[LW_EXTS] = ws[LW_NOPS] = 0;
    const int S = a.alpha * a.alpha + 2;
    for (int k = 0; k < S; ++k)
        a.counts[(int64_t)pid * S + k] = 0;
}

// One wave per pair; the walk's rules are those of kernels.hip's walks.
template <int R>
__global__ __launch_bounds__(64) void kLong16Walk(LongArgs a)
{
    __shared__ int32_t sCnt[16];
    const int slot = blockIdx.x, x = slot & 1, t = threadIdx.x;
    const LongCouple cp = a.couples[slot >> 1];
    int32_t *ws = a.walk + (int64_t)slot * kLongWalkInts;
    if (ws[LW_DONE])
        return;   // the same for every lane
    const int pid = cp.pid[x], p = cp.p[x], A = a.alpha, S = A * A + 2;
    const uint8_t *h = a.hRes + a.hOff[pid], *v = a.vRes + a.vOff[pid];
    if (t < 16)
        sCnt[t] = 0;
    __syncthreads();
    auto field = [&](int k) { return __builtin_amdgcn_readfirstlane(ws[k]); };
    int i = field(LW_I), j = field(LW_J), mode = field(LW_MODE), prev = field(LW_PREV);
    int opens = field(LW_OPENS), exts = field(LW_EXTS), nOps = field(LW_NOPS);
    const Window win = windowOf<R>(p, i, j);
    const int strips = longWinStrips(R), per = strips * kWinCouples;
    const LongRec<R> *rec = reinterpret_cast<const LongRec<R> *>(a.trace) + (int64_t)slot * per * kLongT * 64;
    // Bits of a cell (trace16.hpp's encoding), or -1 outside the window.
    auto bits = [&](int ii, int jj) -> int {
        const int r = p + ii, b = r / (64 * R), rr = r % (64 * R), l = rr / R, k = rr % R;
        const int s = jj + l, c = s / kLongT, u = s % kLongT;
        const int db = win.b0 - b, dc = win.c0 - c;
        if (db < 0 || db >= strips || dc < 0 || dc >= kWinChunks)
            return -1;
        const LongRec<R> &q = rec[((int64_t)(db * kWinCouples + dc / 2) * kLongT + u) * 64 + l];
        const uint32_t ef = q.w[R == 16 ? k >> 3 : 0], dx = q.w[R == 16 ? 2 + (k >> 3) : 1];
        const int sh = (k & 7) + 8 * (dc & 1);
        return (int)(((ef >> sh) & 1u) | (((ef >> (sh + 16)) & 1u) << 1) | (((dx >> sh) & 1u) << 2) |
                     (((dx >> (sh + 16)) & 1u) << 3));
    };
    uint8_t *opEnd = a.ops ? a.ops + a.opOff[pid + 1] : nullptr;
    auto emit = [&](int kind, int k) {   // a run of k equal moves: 0 aligned pairs, 1 gap in H, 2 gap in V
        if (k <= 0)
            return;
        if (kind > 0) {
            opens += prev == kind ? 0 : 1;
            exts += prev == kind ? k : k - 1;
        }
        prev = kind;
        if (opEnd)
            for (int q = t; q < k; q += 64)
                opEnd[-1 - (int64_t)nOps - q] = kind == 0 ? 'M' : kind == 1 ? 'V' : 'H';
        nOps += k;
    };
    bool inside = true;
    while (inside && i > 0 && j > 0) {
        if (mode == 0) {
            const int ii = i - t, jj = j - t;
            // The residues with the bits: one wait instead of two.
            const bool valid = ii > 0 && jj > 0;
            const int rh = valid ? h[jj - 1] : 0, rw = valid ? v[ii - 1] : 0;
            const int b = valid ? bits(ii, jj) : -1;
            const int d = b < 0 ? 3 : (b & 4) ? ((b & 8) ? 2 : 1) : 0;
            const uint64_t other = __ballot(d != 0);
            const int r = other ? __builtin_ctzll(other) : 64;
            if (t < r)
                atomicAdd(&sCnt[min(rh, A - 1) * A + min(rw, A - 1)], 1);
            emit(0, r);
            i -= r;
            j -= r;
            if (r < 64 && i > 0 && j > 0) {
                mode = __builtin_amdgcn_readlane(d, r);
                if (mode == 3) {
                    mode = 0;
                    inside = false;
                }
            }
        } else {
            // A gap: up to the cell that opened it, or row / column 1.
            const bool vert = mode == 1;
            const int gi = vert ? i - t : i, gj = vert ? j : j - t, at = vert ? gi : gj;
            const int b = at > 0 ? bits(gi, gj) : -1;
            const bool ends = b >= 0 && (a.linear || a.alwaysOpen || (b & (vert ? 2 : 1)) != 0 || at == 1);
            const uint64_t any = __ballot(ends || b < 0);
            const int g = any ? __builtin_ctzll(any) : 64;
            const bool stopHere = g < 64 && __builtin_amdgcn_readlane((int)ends, g) != 0;
            inside = g == 64 || stopHere;
            const int len = g + (stopHere ? 1 : 0);
            emit(mode, len);
            if (vert)
                i -= len;
            else
                j -= len;
            if (stopHere)
                mode = 0;
        }
    }
    const bool done = i == 0 || j == 0;
    if (done) {
        // Leading gaps down to the origin (dp_traceback_impl.h:522-545).
        emit(1, i);
        emit(2, j);
    }
    __syncthreads();
    int32_t *cnt = a.counts + (int64_t)pid * S;
    if (t < A * A && sCnt[t])
        cnt[t] += sCnt[t];
    if (t == 0) {
        if (done) {
            cnt[A * A] = opens;
            cnt[A * A + 1] = exts;
            if (a.ops)
                a.opLen[pid] = nOps;
        }
        ws[LW_I] = i;
        ws[LW_J] = j;
        ws[LW_MODE] = mode;
        ws[LW_PREV] = prev;
        ws[LW_OPENS] = opens;
        ws[LW_EXTS] = exts;
        ws[LW_NOPS] = nOps;
        ws[LW_DONE] = done;
    }
}

const void *longKernel(int R)
{
    return R == 16 ? (const void *)&kLong16<16> : R == 8 ? (const void *)&kLong16<8> : (const void *)&kLong16<4>;
}

hipError_t launch(const void *k, int grid, int block, LongArgs args, hipStream_t stream)
{
    void *params[] = {&args};
    return hipLaunchKernel(k, dim3(grid), dim3(block), params, 0, stream);
}

}  // namespace

hipError_t launchLong16(int R, const LongArgs &args, int numCUs, hipStream_t stream)
{
    if (args.nUnits <= 0)
        return hipSuccess;
    return launch(longKernel(R), std::min(numCUs, (args.nUnits + 3) / 4), 64 * kLongWaves, args, stream);
}

hipError_t launchLong16WalkInit(const LongArgs &args, hipStream_t stream)
{
    return launch((const void *)&kLong16WalkInit, (2 * args.nCouples + 63) / 64, 64, args, stream);
}

hipError_t launchLong16Round(int R, const LongArgs &args, hipStream_t stream)
{
    const int blocks = (2 * args.nCouples + 7) / 8 * 8 * longWinBlocks(R);
    const void *tr = R == 16 ? (const void *)&kLong16Trace<16> : R == 8 ? (const void *)&kLong16Trace<8> : (const void *)&kLong16Trace<4>;
    const void *wk = R == 16 ? (const void *)&kLong16Walk<16> : R == 8 ? (const void *)&kLong16Walk<8> : (const void *)&kLong16Walk<4>;
    const hipError_t e = launch(tr, blocks, 256, args, stream);
    return e != hipSuccess ? e : launch(wk, 2 * args.nCouples, 64, args, stream);
}

}  // namespace sqmi
