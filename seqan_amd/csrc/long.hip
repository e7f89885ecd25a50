// long.hip -- int32 kernels for long pairs (global alignment, DNA profile):
// the tiled forward that keeps every tile border as a checkpoint, and the
// checkpointed traceback that recomputes one tile per pair at a time.
//
// The recurrence, borders and traceback decisions are those of the packed
// kernels (kernels.hip), in int32: SeqAn 2's Gotoh formula
// (include/seqan/align/dp_formula_affine.h:62-126), the global borders
// (dp_formula_affine.h:244-330), the trace decisions with the tie rules of
// _maxScore (dp_formula.h:165-201), and the walk of dp_traceback_impl.h:
// 115-546 counted like computeAlignmentStats (evaluate_alignment.h:215-300).
//
// A tile is kTileRows rows (one row block of the pair, bottom-aligned) by
// tileC columns.  One group of 16 lanes sweeps a tile: lane l owns rows
// 16 l .. 16 l + 15 of the block and handles column c0 - 1 + s - l at step s
// (a skewed wavefront; the cell above the lane's first row comes from lane
// l - 1 by DPP row_shr:1, lane 0 reads the block above from the row
// checkpoint).  Inputs: the left column (G = H + gapOpen and E of the
// block's rows at column c0 - 1) and the top row (G and F of the block
// above at columns c0 - 1 .. c1).  Outputs: the bottom row and the right
// column (forward), or 8-byte trace records per lane and step (traceback).
#include "kernels.hpp"
#include "seqan_amd.h"

namespace sqmi {
namespace {

constexpr int kNegL = -(1 << 29);   // minus infinity; real values stay far above
constexpr int TG = 16;              // lanes per group
constexpr int TR = kTileRows / TG;  // rows per lane
constexpr int TQD = 4;              // steps per unrolled loop body
constexpr int TK = 32;              // steps per refill of a group's LDS rings
constexpr int TRING = 64;           // ring entries (two refills)

// Per-group LDS rings of the tile sweep.  top[s % TRING]: the block above's
// bottom row (G, F) at column c0 - 1 + s (lane 0's top input at step s);
// pr[x % TRING]: the substitution profile word of column c0 - 1 + x - 15
// (lane l reads entry s - l + 15 at step s).  Both are refilled every TK
// steps from loads issued TK steps earlier, so the sweep itself issues no
// global loads.
struct GroupRings {
    int2 top[TRING];
    uint32_t pr[TRING];
};

__device__ __forceinline__ int shiftIn16(int v, int first)
{
    return __builtin_amdgcn_update_dpp(first, v, 0x111, 0xf, 0xf, false);
}

__device__ __forceinline__ int subSat32(int a, int b) { return __builtin_elementwise_sub_sat(a, b); }

// Bit k of 32-bit mask pairs: (1 << k) | (1 << (16 + k)).
__device__ __forceinline__ uint32_t rowBits(int k) { return 0x00010001u << k; }

struct TileGeom {
    int b, t;            // row block and column tile
    int c0, c1;          // columns c0 .. c1 of the tile (1-based)
    bool active;         // group has a tile to sweep
};

// One tile sweep for the lane's group.  TRACE: write trace records instead
// of the forward outputs.  HEAD: the tile may hold rows above the pair's row
// 0 (block 0), which are floored at -inf (row 0 at 0 under a free top).
// LOCAL: Smith-Waterman (every H floored at 0, free borders), the maximum G
// of the tile's cells folded into the block's slot of a.best.  The other AlignConfigs
// (forward only): a free left border starts every row at H = 0; the free
// last row and column are reduced from the checkpoints afterwards.
template <bool HEAD, bool TRACE, bool LOCAL = false>
__device__ __forceinline__ void tileSweep(const TileArgs &a, const LongPair &P, const TileGeom &g, int l,
                                          const uint32_t *sProf, GroupRings *rg, uint2 *rec)
{
    const int o = a.gapOpen, e = a.gapExtend, eo = max(o, e);
    const bool leftFree = !TRACE && (LOCAL || (a.mode & SQMI_FREE_LEFT));
    const bool topFree = !TRACE && (a.mode & SQMI_FREE_TOP);
    const int C = a.tileC;
    const uint8_t *h = a.hRes + a.hOff[P.pid];
    const uint8_t *v = a.vRes + a.vOff[P.pid];
    const int n = P.n, m = P.m;
    const int rowbase = g.b * kTileRows + l * TR;
    int32_t *ck = a.ck;
    const int64_t rowIn = P.rowck + ((int64_t)(g.b - 1) * (n + 1)) * 2;   // block b - 1's bottom row
    const int64_t rowOut = P.rowck + ((int64_t)g.b * (n + 1)) * 2;
    const int64_t colIn = P.colck + (((int64_t)g.b * P.ntiles + (g.t - 1)) * kTileRows + l * TR) * 2;
    const int64_t colOut = P.colck + (((int64_t)g.b * P.ntiles + g.t) * kTileRows + l * TR) * 2;

    uint32_t sel[TR];
    int Gk[TR], Ek[TR];
    int floorK[HEAD && !LOCAL ? TR : 1];
#pragma unroll
    for (int k = 0; k < TR; ++k) {
        const int i = rowbase + k - P.p;
        int code = 4;
        if (i >= 1 && i <= m)
            code = min((int)v[i - 1], 4);
        sel[k] = code < 4 ? (0x0c0c0c00u | (uint32_t)code) : 0x0d0d0d0cu;   // pad: t = -256
        if constexpr (HEAD && !LOCAL)
            floorK[k] = (i == 0 && topFree) ? 0 : kNegL;
        if (g.t == 0) {
            // Column 0: -inf above row 0 (local: 0), H(0,0) = 0, then the gap
            // chain growing by max(o, e) per row (free left border: H = 0).
            Gk[k] = (i < 0) ? (LOCAL ? o : kNegL) : (i == 0 || leftFree) ? o : (o + (i - 1) * eo) + o;
            Ek[k] = kNegL;
        } else if (g.active) {
            Gk[k] = ck[colIn + 2 * k];
            Ek[k] = ck[colIn + 2 * k + 1];
        } else {
            Gk[k] = kNegL;
            Ek[k] = kNegL;
        }
    }
    // Top input of the group head at column c0 - 1 + s (the bottom row of
    // block b - 1).  The loads are unconditional: columns past c1 read column
    // c1, and block 0 (no block above) reads its own output row; those values
    // are replaced by -inf.
    const int32_t *topRow = ck + (g.b > 0 ? rowIn : rowOut);
    const bool topReal = g.b > 0 && g.active;
    auto topLoad = [&](int col) -> int2 { return *reinterpret_cast<const int2 *>(topRow + 2 * min(col, g.c1)); };
    if (!TRACE && g.active && g.t == 0 && l == TG - 1)
        *reinterpret_cast<int2 *>(ck + rowOut) = make_int2(Gk[TR - 1], kNegL);   // column 0 of the bottom row

    int botG = Gk[TR - 1], botF = kNegL;
    int upGprev = kNegL;
    int bestG = o;   // local: H = 0, the empty alignment
    const int width = g.c1 - g.c0 + 1;
    const int steps = ((width + TG + TQD - 1) / TQD) * TQD;
    // Ring refills: the refill for steps [s, s + TK) covers columns
    // c0 - 1 + s + 2 l and + 1 of lane l (top entries s + 2 l, profile
    // entries s + 15 + 2 l); residue indexes are clamped into H (columns
    // outside it are never computed).
    auto hLoad = [&](int col) -> uint32_t { return (uint32_t)h[min(max(col, 1), n) - 1]; };
    int2 t0, t1;
    uint32_t h0, h1;
    auto refillLoad = [&](int s) {
        const int cb = g.c0 - 1 + s + 2 * l;
        t0 = topLoad(cb);
        t1 = topLoad(cb + 1);
        h0 = hLoad(cb);
        h1 = hLoad(cb + 1);
    };
    auto refillStore = [&](int s) {
        rg->top[(s + 2 * l) & (TRING - 1)] = t0;
        rg->top[(s + 2 * l + 1) & (TRING - 1)] = t1;
        rg->pr[(s + TG - 1 + 2 * l) & (TRING - 1)] = sProf[min(h0, 4u)];
        rg->pr[(s + TG + 2 * l) & (TRING - 1)] = sProf[min(h1, 4u)];
        __builtin_amdgcn_wave_barrier();
    };
    refillLoad(0);
    refillStore(0);
    refillLoad(TK);
    uint32_t prof = rg->pr[(TG - 1 - l) & (TRING - 1)];
    int2 topv = rg->top[0];

    auto step = [&](int s, uint32_t pr, int2 top) {
        const int jj = g.c0 - 1 + s - l;
        const bool topOk = topReal && g.c0 - 1 + s <= g.c1;
        const int upG = shiftIn16(botG, topOk ? top.x : kNegL);
        const int upF = shiftIn16(botF, topOk ? top.y : kNegL);
        const int diagTop = upGprev;
        upGprev = upG;
        if (jj >= g.c0 && jj <= g.c1) {
            int uG = upG, uF = upF;
            uint32_t accEF = 0, accDX = 0;
            // D: the diagonal term of row k, H(i-1, j-1) + s(h, v), taken
            // from the old G of row k - 1 before it is overwritten.
            int D = diagTop + (int)__builtin_amdgcn_perm(0u, pr, sel[0]);
#pragma unroll
            for (int k = 0; k < TR; ++k) {
                const int Eext = Ek[k] + e, Fext = uF + e;
                const int Gleft = Gk[k];
                const int E = max(Eext, Gleft);
                const int F = max(Fext, uG);
                int H;
                if constexpr (TRACE) {
                    // Sign bytes of the decisions: E opened, F opened (bits k,
                    // 16 + k of accEF); not diagonal, E beats F (accDX).
                    const uint32_t ef = __builtin_amdgcn_perm((uint32_t)subSat32(Fext, uG),
                                                              (uint32_t)subSat32(Eext, Gleft), 0x0b0b0909u);
                    const int fe = max(E, F);
                    const uint32_t dx = __builtin_amdgcn_perm((uint32_t)subSat32(F, E),
                                                              (uint32_t)subSat32(D, fe), 0x0b0b0909u);
                    H = max(D, fe);
                    const uint32_t bit = rowBits(k);
                    asm volatile("v_bfi_b32 %0, %1, %2, %0" : "+v"(accEF) : "s"(bit), "v"(ef));
                    asm volatile("v_bfi_b32 %0, %1, %2, %0" : "+v"(accDX) : "s"(bit), "v"(dx));
                } else {
                    H = max(D, max(E, F));
                }
                if constexpr (LOCAL)
                    H = max(H, 0);
                else if constexpr (HEAD)
                    H = max(H, floorK[k]);
                if (k + 1 < TR)
                    D = Gleft + (int)__builtin_amdgcn_perm(0u, pr, sel[k + 1]);
                Ek[k] = E;
                Gk[k] = H + o;
                if constexpr (LOCAL)
                    bestG = max(bestG, Gk[k]);
                uG = Gk[k];
                uF = F;
            }
            botG = uG;
            botF = uF;
            if (g.active) {
                if constexpr (TRACE) {
                    rec[s * TG + l] = make_uint2(accEF, accDX);
                } else {
                    if (l == TG - 1)
                        *reinterpret_cast<int2 *>(ck + rowOut + 2 * jj) = make_int2(botG, botF);
                    // The right column (the last tile's too: a free last
                    // column is reduced from it).
                    if (jj == g.c1) {
#pragma unroll
                        for (int k = 0; k < TR; ++k)
                            *reinterpret_cast<int2 *>(ck + colOut + 2 * k) = make_int2(Gk[k], Ek[k]);
                    }
                    // Cell (m, n): the last row of the last block.
                    if (l == TG - 1 && jj == n && g.b == P.nblocks - 1) {
                        a.scores[P.pid] = botG - o;
                        a.endEF[2 * P.pid] = Ek[TR - 1];
                        a.endEF[2 * P.pid + 1] = botF;
                    }
                }
            }
        }
    };
    for (int s0 = 0; s0 < steps; s0 += TQD) {
        if ((s0 & (TK - 1)) == TK - TQD) {
            // Rings for the next TK steps (read from the next step on), and
            // the loads for the refill after it.
            refillStore(s0 + TQD);
            refillLoad(s0 + TQD + TK);
        }
#pragma unroll
        for (int u = 0; u < TQD; ++u) {
            const int s = s0 + u;
            const uint32_t prN = rg->pr[(s + 1 + TG - 1 - l) & (TRING - 1)];
            const int2 topN = rg->top[(s + 1) & (TRING - 1)];
            step(s, prof, topv);
            prof = prN;
            topv = topN;
        }
    }
    if constexpr (LOCAL) {
        // The group's maximum into the block's slot: one tile of a block per
        // launch, so the slot has no other writer (its first tile starts it).
#pragma unroll
        for (int d = 1; d < TG; d <<= 1)
            bestG = max(bestG, __shfl_xor(bestG, d, TG));
        if (g.active && l == 0) {
            int32_t *slot = a.best + P.bestck + g.b;
            *slot = g.t == 0 ? bestG : max(*slot, bestG);
        }
    }
}

__device__ __forceinline__ void loadProfile(const TileArgs &a, uint32_t *sProf)
{
    if (threadIdx.x < 5)
        sProf[threadIdx.x] = a.dnaProfile[threadIdx.x];
    __syncthreads();
}

// Forward: the tiles of anti-diagonal a.diag.  Each wave takes four
// consecutive row blocks of one pair (one per 16-lane group).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void kTileFwd32(TileArgs a)
{
    __shared__ uint32_t sProf[8];
    __shared__ GroupRings sRings[256 / TG];
    loadProfile(a, sProf);
    const int lane = threadIdx.x & 63, l = lane % TG, grp = lane / TG;
    const int w = blockIdx.x * (blockDim.x >> 6) + (int)(threadIdx.x >> 6);
    const int pi = w / a.wavesPerPair;
    if (pi >= a.nPairs)
        return;
    const LongPair P = a.pairs[pi];
    const int b0 = (w % a.wavesPerPair) * 4;
    TileGeom g;
    g.b = b0 + grp;
    g.t = a.diag - g.b;
    g.active = g.b < P.nblocks && g.t >= 0 && g.t < P.ntiles;
    if (!__any(g.active))
        return;   // the whole wave is idle on this diagonal
    if (!g.active) {
        g.b = min(g.b, P.nblocks - 1);
        g.t = min(max(g.t, 0), P.ntiles - 1);
    }
    g.c0 = g.t * a.tileC + 1;
    g.c1 = min((g.t + 1) * a.tileC, P.n);
    if (a.mode & SQMI_LOCAL) {
        tileSweep<false, false, true>(a, P, g, l, sProf, &sRings[threadIdx.x / TG], nullptr);
    } else if (b0 == 0) {
        tileSweep<true, false>(a, P, g, l, sProf, &sRings[threadIdx.x / TG], nullptr);
    } else {
        tileSweep<false, false>(a, P, g, l, sProf, &sRings[threadIdx.x / TG], nullptr);
    }
}

// Walk state of one long pair: the cell (i, j) reached, the walk mode
// (0: choose from the cell's H decision, 1 / 2: inside a vertical /
// horizontal gap), the last operation, gap opens / extensions, done flag.
enum { WS_I = 0, WS_J, WS_MODE, WS_PREV, WS_OPENS, WS_EXTS, WS_DONE, WS_NOPS };

__device__ __forceinline__ TileGeom walkTile(const TileArgs &a, const LongPair &P, const int32_t *ws)
{
    TileGeom g;
    const int i = ws[WS_I], j = ws[WS_J];
    g.active = ws[WS_DONE] == 0 && i > 0 && j > 0;
    const int ii = g.active ? i : P.m, jj = g.active ? j : P.n;
    g.b = (P.p + ii) / kTileRows;
    g.t = (jj - 1) / a.tileC;
    g.c0 = g.t * a.tileC + 1;
    g.c1 = min((g.t + 1) * a.tileC, P.n);
    return g;
}

// Traceback rounds.  A round recomputes, with trace records, the window of
// kRoundBlocks x kRoundTiles tiles whose bottom-right tile holds the walk's
// position (every tile of it only needs checkpoints, so all of them run at
// once), then walks the pair through the window.  The walk leaves a window
// through its top or left side, so each round moves it up kRoundBlocks row
// blocks or left kRoundTiles tiles.

// Window slot of tile (b, t) for a window whose bottom-right tile is (b0, t0).
__device__ __forceinline__ int windowSlot(int b0, int t0, int b, int t) { return (b0 - b) * kRoundTiles + (t0 - t); }

// Step 1: one 16-lane group per (pair, window slot).  Workgroup w serves
// pairs with the same w mod 8 (the walk of pair p runs in workgroup p, and
// workgroups are spread over the 8 XCDs by id mod 8, so both kernels of a
// pair share one L2).
constexpr int kTraceGroupsPerWG = 16;
constexpr int kTraceWGsPerPair = kRoundSlots / kTraceGroupsPerWG;
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void kTileTrace32(TileArgs a)
{
    __shared__ uint32_t sProf[8];
    __shared__ GroupRings sRings[256 / TG];
    loadProfile(a, sProf);
    const int lane = threadIdx.x & 63, l = lane % TG;
    const int w = blockIdx.x;
    const int pi = 8 * (w / (8 * kTraceWGsPerPair)) + (w % 8);
    const int slot = ((w / 8) % kTraceWGsPerPair) * kTraceGroupsPerWG + (int)(threadIdx.x / TG);
    const bool exists = pi < a.nPairs;
    const int pc = exists ? pi : a.nPairs - 1;
    const LongPair P = a.pairs[pc];
    TileGeom g = walkTile(a, P, a.walk + (int64_t)pc * kWalkStateInts);
    g.b -= slot / kRoundTiles;
    g.t -= slot % kRoundTiles;
    g.active = g.active && exists && g.b >= 0 && g.t >= 0;
    if (!__any(g.active))
        return;
    if (!g.active) {
        g.b = max(g.b, 0);
        g.t = max(g.t, 0);
    }
    g.c0 = g.t * a.tileC + 1;
    g.c1 = min((g.t + 1) * a.tileC, P.n);
    uint2 *rec = a.trace + ((int64_t)pc * kRoundSlots + slot) * kTileRecSteps * TG;
    tileSweep<true, true>(a, P, g, l, sProf, &sRings[threadIdx.x / TG], rec);
}

__global__ void kTileWalkInit(TileArgs a)
{
    const int pi = blockIdx.x * blockDim.x + threadIdx.x;
    if (pi >= a.nPairs)
        return;
    const LongPair P = a.pairs[pi];
    int32_t *ws = a.walk + (int64_t)pi * kWalkStateInts;
    const int score = a.scores[P.pid], endE = a.endEF[2 * P.pid], endF = a.endEF[2 * P.pid + 1];
    ws[WS_I] = P.m;
    ws[WS_J] = P.n;
    // End cell: F, then E, win ties (dp_algorithm_impl.h:1190-1207,
    // PreferGapsAtEnd_ dp_traceback_impl.h:115-122); the linear-gap walk
    // (gap open == gap extend) takes the cell's own direction.
    ws[WS_MODE] = (a.gapOpen == a.gapExtend) ? 0 : (endF == score) ? 1 : (endE == score) ? 2 : 0;
    ws[WS_PREV] = 0;
    ws[WS_OPENS] = 0;
    ws[WS_EXTS] = 0;
    ws[WS_DONE] = 0;
    ws[WS_NOPS] = 0;
    const int S = a.alpha * a.alpha + 2;
    for (int k = 0; k < S; ++k)
        a.counts[(int64_t)P.pid * S + k] = 0;
}

// Step 2: one workgroup per pair walks it through the window.  The records
// of half a tile (128 rows: lanes 0-7 or 8-15 of the sweep) are staged in
// LDS by the whole workgroup; thread 0 walks them, and the next half tile is
// staged when the walk leaves this one.
constexpr int kWalkWGThreads = 256;
constexpr int kHalfLanes = TG / 2;
__global__ __launch_bounds__(kWalkWGThreads) void kTileWalk32(TileArgs a)
{
    __shared__ uint2 sRec[kTileRecSteps * kHalfLanes];
    __shared__ uint8_t sH[kLongTileC], sV[kTileRows / 2];   // residues of the half tile's columns and rows
    __shared__ int32_t sCnt[16];
    __shared__ int32_t sUnit[4];   // b, t, half, stop
    const int pi = blockIdx.x;
    if (pi >= a.nPairs)
        return;
    const LongPair P = a.pairs[pi];
    int32_t *ws = a.walk + (int64_t)pi * kWalkStateInts;
    const TileGeom g0 = walkTile(a, P, ws);
    if (!g0.active)
        return;   // finished (the same for every thread of the workgroup)
    const int A = a.alpha, S = A * A + 2;
    const bool linear = a.gapOpen == a.gapExtend;
    const uint8_t *h = a.hRes + a.hOff[P.pid];
    const uint8_t *v = a.vRes + a.vOff[P.pid];
    const int tid = threadIdx.x;
    if (tid < 16)
        sCnt[tid] = 0;
    int i = 0, j = 0, mode = 0, prev = 0, opens = 0, exts = 0, nOps = 0;
    if (tid == 0) {
        i = ws[WS_I];
        j = ws[WS_J];
        mode = ws[WS_MODE];
        prev = ws[WS_PREV];
        opens = ws[WS_OPENS];
        exts = ws[WS_EXTS];
        nOps = ws[WS_NOPS];
    }
    // Rows: written backwards from the end of the pair's op segment.
    uint8_t *opEnd = a.ops ? a.ops + a.opOff[P.pid + 1] : nullptr;
    auto emit = [&](uint8_t op) {
        if (opEnd)
            opEnd[-1 - (int64_t)nOps] = op;
        ++nOps;
    };
    for (;;) {
        if (tid == 0) {
            // The unit (tile, half) holding (i, j), or stop: finished or
            // outside the window.
            const int b = (P.p + i) / kTileRows, t = (j - 1) / a.tileC;
            const int half = ((P.p + i) % kTileRows) / (kTileRows / 2);
            const bool inside = i > 0 && j > 0 && b <= g0.b && b > g0.b - kRoundBlocks && t <= g0.t &&
                                t > g0.t - kRoundTiles;
            sUnit[0] = b;
            sUnit[1] = t;
            sUnit[2] = half;
            sUnit[3] = inside ? 0 : 1;
        }
        __syncthreads();
        const int ub = sUnit[0], ut = sUnit[1], uh = sUnit[2];
        if (sUnit[3])
            break;
        // Stage the half tile: records rec[s * 16 + 8 * half + 0..7] for all steps.
        const uint2 *rec = a.trace + ((int64_t)pi * kRoundSlots + windowSlot(g0.b, g0.t, ub, ut)) * kTileRecSteps * TG;
        const uint4 *src = reinterpret_cast<const uint4 *>(rec);
        uint4 *dst = reinterpret_cast<uint4 *>(sRec);
        for (int x = tid; x < kTileRecSteps * kHalfLanes / 2; x += kWalkWGThreads) {
            const int st = x / (kHalfLanes / 2), c = x % (kHalfLanes / 2);
            dst[x] = src[st * (TG / 2) + uh * (kHalfLanes / 2) + c];
        }
        const int c0 = ut * a.tileC + 1;
        const int rowTop = ub * kTileRows + uh * (kTileRows / 2) - P.p;   // first pair row of the half
        for (int x = tid; x < a.tileC; x += kWalkWGThreads)
            sH[x] = h[min(c0 + x, P.n) - 1];
        if (tid < kTileRows / 2)
            sV[tid] = v[min(max(rowTop + tid, 1), P.m) - 1];
        __syncthreads();
        if (tid == 0) {
            while (i > 0 && j > 0 && i >= rowTop && j >= c0) {
                const int r = P.p + i - ub * kTileRows;
                const int l = r / TR, k = r % TR;
                const uint2 w = sRec[(j - (c0 - 1) + l) * kHalfLanes + (l - uh * kHalfLanes)];
                const uint32_t sh = (uint32_t)k;
                const uint32_t bits = ((w.x >> sh) & 1u) | (((w.x >> (sh + 16)) & 1u) << 1) |
                                      (((w.y >> sh) & 1u) << 2) | (((w.y >> (sh + 16)) & 1u) << 3);
                const int d = mode == 0 ? ((bits & 4u) ? ((bits & 8u) ? 2 : 1) : 0) : mode;
                if (d == 0) {
                    const int hc = min((int)sH[j - c0], A - 1), vc = min((int)sV[i - rowTop], A - 1);
                    sCnt[hc * A + vc] += 1;
                    emit('M');
                    prev = 0;
                    --i;
                    --j;
                    mode = 0;
                } else {
                    // One gap character; the gap goes on while the cell's gap
                    // extends, down to row / column 1 (dp_traceback_impl.h:220-341).
                    // Linear gaps (gap open == gap extend) take one step per
                    // cell and re-read the next cell's own direction.
                    const bool vert = d == 1;
                    const bool open = (bits & (vert ? 2u : 1u)) != 0;
                    if (prev == d) ++exts; else ++opens;
                    prev = d;
                    emit(vert ? 'V' : 'H');
                    const bool stop = linear || open || (vert ? i == 1 : j == 1);
                    if (vert)
                        --i;
                    else
                        --j;
                    mode = stop ? 0 : d;
                }
            }
        }
        __syncthreads();   // sRec is restaged next
    }
    if (tid == 0) {
        int32_t *cnt = a.counts + (int64_t)P.pid * S;
        for (int k = 0; k < A * A; ++k)
            if (sCnt[k])
                cnt[k] += sCnt[k];
        if (i == 0 || j == 0) {
            // Leading gaps down to the origin (dp_traceback_impl.h:522-545).
            if (i > 0) {
                if (prev == 1) exts += i; else { ++opens; exts += i - 1; }
                prev = 1;
                for (int k = 0; k < i; ++k)
                    emit('V');
            }
            if (j > 0) {
                if (prev == 2) exts += j; else { ++opens; exts += j - 1; }
                for (int k = 0; k < j; ++k)
                    emit('H');
            }
            cnt[A * A] += opens;
            cnt[A * A + 1] += exts;
            if (a.ops)
                a.opLen[P.pid] = nOps;
            ws[WS_DONE] = 1;
        }
        ws[WS_I] = i;
        ws[WS_J] = j;
        ws[WS_MODE] = mode;
        ws[WS_PREV] = prev;
        ws[WS_OPENS] = opens;
        ws[WS_EXTS] = exts;
        ws[WS_NOPS] = nOps;
    }
}

}  // namespace

// Results of long pairs under free end gaps or local alignment, one
// workgroup per pair: the maximum G over the cells the AlignConfig tracks
// (dp_scout.h:169-210; the reference's own scouts, restated in the oracle):
// the last row (free bottom: the last block's bottom-row checkpoint, columns
// 0 .. n), the last column (free right: the last tile's right-column
// checkpoints, rows 0 .. m), or every cell (local: the maxima of the row
// blocks the tile sweeps kept).  Score = G - gapOpen.
__global__ __launch_bounds__(256) void kLongResult(TileArgs a)
{
    __shared__ int red[256 / 64];
    const int pi = blockIdx.x;
    if (pi >= a.nPairs)
        return;
    const LongPair P = a.pairs[pi];
    const int32_t *ck = a.ck;
    const bool local = (a.mode & SQMI_LOCAL) != 0;
    int best = kNegL;
    if (local) {
        for (int b = threadIdx.x; b < P.nblocks; b += blockDim.x)
            best = max(best, a.best[P.bestck + b]);
    }
    if (!local && (a.mode & SQMI_FREE_BOTTOM)) {
        const int64_t row = P.rowck + (int64_t)(P.nblocks - 1) * (P.n + 1) * 2;
        for (int j = threadIdx.x; j <= P.n; j += blockDim.x)
            best = max(best, ck[row + 2 * j]);
    }
    if (!local && (a.mode & SQMI_FREE_RIGHT)) {
        for (int r = threadIdx.x; r < P.nblocks * kTileRows; r += blockDim.x) {
            const int i = r - P.p;
            if (i >= 0 && i <= P.m)
                best = max(best, ck[P.colck + (((int64_t)(r / kTileRows) * P.ntiles + (P.ntiles - 1)) * kTileRows +
                                               r % kTileRows) * 2]);
        }
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
        best = max(best, __shfl_xor(best, d, 64));
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
            best = max(best, red[w]);
        if (local || (a.mode & (SQMI_FREE_BOTTOM | SQMI_FREE_RIGHT)))
            a.scores[P.pid] = best - a.gapOpen;
    }
}

hipError_t launchLongResult(const TileArgs &args, hipStream_t stream)
{
    if (args.nPairs <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(kLongResult, dim3(args.nPairs), dim3(256), 0, stream, args);
    return hipGetLastError();
}

hipError_t launchTileFwd32(const TileArgs &args, hipStream_t stream)
{
    const int waves = args.nPairs * args.wavesPerPair;
    if (waves <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(kTileFwd32, dim3((waves + 3) / 4), dim3(256), 0, stream, args);
    return hipGetLastError();
}

hipError_t launchTileTrace32(const TileArgs &args, hipStream_t stream)
{
    if (args.nPairs <= 0)
        return hipSuccess;
    const int wgs = ((args.nPairs + 7) / 8) * 8 * kTraceWGsPerPair;
    hipLaunchKernelGGL(kTileTrace32, dim3(wgs), dim3(256), 0, stream, args);
    return hipGetLastError();
}

hipError_t launchTileWalkInit(const TileArgs &args, hipStream_t stream)
{
    if (args.nPairs <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(kTileWalkInit, dim3((args.nPairs + 63) / 64), dim3(64), 0, stream, args);
    return hipGetLastError();
}

hipError_t launchTileWalk32(const TileArgs &args, hipStream_t stream)
{
    if (args.nPairs <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(kTileWalk32, dim3(args.nPairs), dim3(kWalkWGThreads), 0, stream, args);
    return hipGetLastError();
}

}  // namespace sqmi
