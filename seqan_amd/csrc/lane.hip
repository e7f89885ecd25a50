// lane.hip -- the one-pair-per-lane form of the packed int16 forward.
//
// The reference's inter-sequence form puts one pair in every SIMD lane and
// pads a batch of 8 / 16 pairs to the batch's maximum lengths
// (include/seqan/align/dp_align_simd_helper.h:147-221, 277-347).  Here every
// lane of a wavefront holds a couple of pairs (the low and high int16 halves
// of its registers), so one wavefront sweeps 128 pairs, and the planner fills
// a wavefront with pairs of nearly one shape (same number of R-row blocks,
// widths sorted), which keeps the padding near zero.
//
// Recurrence, borders and result cells are those of the packed family
// (kernels.hip, G-space Gotoh of include/seqan/align/dp_formula_affine.h:
// 62-126 with the tracking rules of dp_meta_info.h:178-221 and
// dp_scout.h:169-210):
//
//   E(i,j) = max(E(i,j-1) + e, G(i,j-1))
//   F(i,j) = max(F(i-1,j) + e, G(i-1,j))
//   H(i,j) = max(G(i-1,j-1) + t(h,v), E(i,j), F(i,j))   [local: max(., 0)]
//   G(i,j) = H(i,j) + o,   t = s - o
//
// Global scores hold drifted values (kernels.hpp, Drift), which make a gap
// step free of additions and keep every value >= 0; local scores hold the
// values themselves and saturate.
//
// A lane sweeps its couple in blocks of R rows (rows bottom-aligned: row m
// is the last row of the last block, the rows above row 0 are virtual), all
// columns of one block before the next.  The virtual rows need no floor:
// under drift they stay at or below minus infinity's stand-in, in the local
// kernels the saturating adds let them sink.  Under a free first row, row 0
// of the first block gains drift per column (H(0, j) = 0).  No value crosses lanes, so there is no
// skew and no lane shift; the bottom row of a block (G, F per column) goes
// to a per-wave row buffer laid out column-major across the 64 lanes (one
// coalesced 512-byte load and store per column), read back by the next
// block.  The row buffer and the residues are loaded one group of QD = 4
// columns ahead of the sweep; the residues as one aligned dword window per
// pair and group.
//
// Substitution scores.  DNA: each row keeps, per pair, the word of t(h, v)
// over h = 0..3 for its residue v (the padding code: zero bytes); each
// column builds one v_perm selector for both pairs from its two residues,
// and one v_perm per row then yields t for both halves.  Other alphabets:
// the (alpha + 1)^2 table in LDS, two reads per cell.
#include "kernels.hpp"
#include "packed16.hpp"
#include "seqan_amd.h"

namespace sqmi {
namespace {

template <int R, bool DNA, uint32_t TRK>
struct Lane16 {
    static constexpr bool LOC = (TRK & kTrackLocal) != 0;
    static constexpr bool WIDE = (TRK & kWideVals) != 0;
    static constexpr int QD = 4;   // columns per group: one dword of residues per pair

    struct Couple {
        const uint8_t *h[2];
        const uint8_t *v[2];
        int n[2], m[2], p[2], pid[2];
    };

    __device__ __forceinline__ static int padded(int Nw) { return (Nw + QD - 1) / QD * QD; }

    // Row-buffer columns a work item of width Nw needs (one group of prefetch
    // past the padded width).
    __host__ __device__ static int rowColsFor(int Nw) { return (Nw + QD - 1) / QD * QD + QD + 1; }

    // Residues of a pair, read as aligned dwords: group g (columns 4g + 1
    // .. 4g + 4, bytes h[4g] .. h[4g + 3]) is the funnel shift by `mis` of
    // dwords g and g + 1 of `words` (the dword-aligned start of the pair's
    // residues).  Both indexes are clamped to `lastW`, the dword holding the
    // pair's last residue, so no read leaves the pages of the pair's own
    // residues; bytes for columns past n are then arbitrary and are masked
    // (local, non-DNA) or cannot reach a result (a column never feeds the
    // columns left of it).
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

    // One block of R rows: column 0, then columns 1 .. Nw (rounded up to QD;
    // the extra columns cannot change a result).  FIRST: block 0, with no
    // row above it (-inf).  TOPFREE: block 0 under a free first row: row 0
    // takes E(0, j) = H(0, j) = E(0, j - 1) + drift.
    template <bool FIRST, bool TOPFREE>
    __device__ __forceinline__ static void block(const FwdArgs &a, const Couple &c, int b, int Nw, bool last,
                                                 uint2 *rb, const uint32_t *sProf, const int16_t *sT, s16x2 &best,
                                                 int2 &bestH)
    {
        const int o = a.gapOpen, e = a.gapExtend;
        const Drift dr = a.drift;
        const s16x2 o2 = splat(o), e2 = splat(e), neg2 = splat(LOC ? kNeg16 : dr.neg);
        // In vector registers: 32-bit adds with scalar operands issue slower.
        uint32_t cost2 = (uint32_t)dr.cost * 0x10001u, d2 = (uint32_t)dr.d * 0x10001u;
        if constexpr (!LOC)
            asm volatile("" : "+v"(cost2), "+v"(d2));
        const bool leftFree = (a.mode & (SQMI_FREE_LEFT | SQMI_LOCAL)) != 0;
        const int eo = max(e, o);   // the first column's gap chain grows by max(e, o) per row
        const int PAD = a.alpha;
        const int TW = a.alpha + 1;
        const int rowbase = b * R;

        // Per row: DNA the row words of both pairs, else the two row codes.
        uint32_t rowA[R], rowB[DNA ? R : 1];
        s16x2 Gk[R], Ek[R];
        uint32_t rowD[TOPFREE ? R : 1];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            int code[2], g0[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int i = rowbase + k - c.p[x];
                int cc = PAD;
                if (i >= 1) {
                    const int idx = min(i - 1, max(c.m[x] - 1, 0));
                    cc = min((int)c.v[x][idx], PAD);
                }
                code[x] = cc;
                // G at column 0: virtual rows -inf, H(0,0) = 0, the first column.
                g0[x] = (i < 0) ? kNeg16 : (i == 0) ? o : ((leftFree ? 0 : o + (i - 1) * eo) + o);
                if constexpr (!LOC)
                    g0[x] = (i < 0) ? dr.neg : (i == 0) ? dr.bias - dr.cost
                            : leftFree ? dr.bias + dr.d * i - dr.cost : dr.bias - 2 * dr.cost;
            }
            if constexpr (DNA) {
                rowA[k] = sProf[8 + code[0]];
                rowB[k] = sProf[8 + code[1]];
            } else {
                rowA[k] = (uint32_t)code[0] | ((uint32_t)code[1] << 16);
            }
            Gk[k] = pack(g0[0], g0[1]);
            Ek[k] = neg2;
            if constexpr (TOPFREE) {
                const uint32_t top = (rowbase + k == c.p[0] ? 0xffffu : 0u) | (rowbase + k == c.p[1] ? 0xffff0000u : 0u);
                rowD[k] = d2 & top;
                Ek[k] = as16(bfi(top, asu(splat(dr.bias)), asu(neg2)));
            }
        }
        // Free last row: the running maximum of the bottom row's stored G,
        // gaining drift per column so that it stays comparable; its true
        // value is taken at column n.
        uint32_t botM = asu(Gk[R - 1]);
        const int base[2] = {dr.cost - dr.bias - dr.d * c.m[0], dr.cost - dr.bias - dr.d * c.m[1]};

        // Column 0 of the previous block's bottom row (the diagonal input of
        // column 1), then this block's own column-0 entry.
        s16x2 upGprev = neg2;
        if constexpr (!FIRST)
            upGprev = as16(rb[0].x);
        if (!last)
            rb[0] = make_uint2(asu(Gk[R - 1]), asu(neg2));

        const int NwP = padded(Nw);
        const s16x2 nHalf = pack(c.n[0], c.n[1]);
        // Row-buffer entries of the next QD columns (blocks after the first),
        // and the residue dwords of the next group, are always in flight.
        uint2 rq[QD];
#pragma unroll
        for (int u = 0; u < QD; ++u)
            rq[u] = FIRST ? make_uint2(asu(neg2), asu(neg2)) : rb[(1 + u) * 64];
        const Residues ra = residues(c.h[0], c.n[0]), rbs = residues(c.h[1], c.n[1]);
        uint32_t a0 = ra.words[min(0, ra.lastW)], a1 = ra.words[min(1, ra.lastW)];
        uint32_t b0 = rbs.words[min(0, rbs.lastW)], b1 = rbs.words[min(1, rbs.lastW)];
        for (int s0 = 1, g = 0; s0 <= NwP; s0 += QD, ++g) {
            const uint32_t curA = __builtin_amdgcn_alignbyte(a1, a0, ra.mis);
            const uint32_t curB = __builtin_amdgcn_alignbyte(b1, b0, rbs.mis);
            // The next group's residue dwords (past the width: unused reads
            // of the clamped dwords).
            a0 = ra.words[min(g + 1, ra.lastW)];
            a1 = ra.words[min(g + 2, ra.lastW)];
            b0 = rbs.words[min(g + 1, rbs.lastW)];
            b1 = rbs.words[min(g + 2, rbs.lastW)];
#pragma unroll
            for (int u = 0; u < QD; ++u) {
                const int j = s0 + u;
                const uint2 up = rq[u];
                // Column j + QD: its row-buffer entry is read before this
                // block writes it (QD steps from now); past the item's width
                // it is an unused in-bounds read.
                if constexpr (!FIRST)
                    rq[u] = rb[(j + QD) * 64];
                // 0xffff in the halves where j > n.
                auto afterMask = [&]() -> uint32_t { return asu((nHalf - splat(j)) >> splat(15)); };
                uint32_t colSel = 0, pA = 0, pB = 0;
                if constexpr (DNA) {
                    // [h_A, 0x0c, h_B + 4, 0x0c]: byte h_A of the pair-A row
                    // word, byte h_B of the pair-B one, zero high bytes.
                    const uint32_t pick = (uint32_t)u | (0x0cu << 8) | ((uint32_t)(4 + u) << 16) | (0x0cu << 24);
                    colSel = __builtin_amdgcn_perm(curB, curA, pick) | 0x0c040c00u;
                    if constexpr (TRK & kTrackLocal)
                        colSel = bfi(afterMask(), 0x0c0c0c0cu, colSel);   // padding columns: t = 0
                } else {
                    const uint32_t after = afterMask();
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
                s16x2 uG = as16(up.x), uF = as16(up.y);
                const s16x2 upG = uG;
                // The diagonal term of row k comes from the old G of row k - 1
                // before it is overwritten.
                auto dOf = [&](s16x2 g, int k) -> s16x2 {
                    if constexpr (LOC)
                        return addSat(g, as16(tOf(k)));
                    else if constexpr (DNA && !WIDE)
                        return as16(asu(g) + tOf(k));   // t >= 0 and halves below 0x8000: no carry
                    else
                        return as16(uadd2(asu(g), tOf(k)));
                };
                s16x2 D = dOf(upGprev, 0);
#pragma unroll
                for (int k = 0; k < R; ++k) {
                    s16x2 F, Gn;
                    if constexpr (LOC) {
                        Ek[k] = vmax(addSat(Ek[k], e2), Gk[k]);
                        F = vmax(addSat(uF, e2), uG);
                        const s16x2 H = vmax(vmax(vmax(D, Ek[k]), F), splat(0));
                        if (k + 1 < R)
                            D = dOf(Gk[k], k + 1);
                        Gn = addSat(H, o2);
                        best = vmax(best, Gn);
                    } else {
                        uint32_t Ev = asu(Ek[k]);
                        if constexpr (TOPFREE)
                            Ev = uadd2(Ev, rowD[k]);
                        Ev = umax2(Ev, asu(Gk[k]));
                        const uint32_t Fv = umax2(asu(uF), asu(uG));
                        const uint32_t H = WIDE ? umax2(umax2(asu(D), Ev), Fv) : max3Pos(asu(D), Ev, Fv);
                        if (k + 1 < R)
                            D = dOf(Gk[k], k + 1);
                        Ek[k] = as16(Ev);
                        F = as16(Fv);
                        Gn = as16(WIDE ? usub2(H, cost2) : H - cost2);
                    }
                    Gk[k] = Gn;
                    uG = Gn;
                    uF = F;
                }
                upGprev = upG;
                if (!last)
                    rb[j * 64] = make_uint2(asu(uG), asu(uF));
                if constexpr (!LOC) {
                    const s16x2 rem = nHalf - splat(j);   // n - j per half
                    if constexpr (TRK & (kTrackEnd | kTrackBottom)) {
                        if (last) {
                            botM = (TRK & kTrackBottom) ? umax2(uadd2(botM, d2), asu(uG)) : asu(uG);
                            if ((uint16_t)rem.x == 0)
                                bestH.x = max(bestH.x, (int)(botM & 0xffffu) + base[0] - dr.d * j);
                            if ((uint16_t)rem.y == 0)
                                bestH.y = max(bestH.y, (int)(botM >> 16) + base[1] - dr.d * j);
                        }
                    }
                    if constexpr (TRK & kTrackRight) {
                        // The maximum of the block's rows in column n, per
                        // half: down the rows the running maximum gains drift
                        // per row; rows above row 0 are left out.
                        if ((uint16_t)rem.x == 0 || (uint16_t)rem.y == 0) {
                            const int iTop[2] = {rowbase - c.p[0], rowbase - c.p[1]};
                            uint32_t mx = asu(Gk[0]);
#pragma unroll
                            for (int k = 1; k < R; ++k) {
                                mx = uadd2(mx, d2);
                                if constexpr (FIRST)
                                    mx &= ~((iTop[0] + k - 1 < 0 ? 0xffffu : 0u) | (iTop[1] + k - 1 < 0 ? 0xffff0000u : 0u));
                                mx = umax2(mx, asu(Gk[k]));
                            }
                            if ((uint16_t)rem.x == 0 && iTop[0] + R > 0)
                                bestH.x = max(bestH.x, (int)(mx & 0xffffu) + dr.cost - dr.bias -
                                                           dr.d * (iTop[0] + R - 1 + j));
                            if ((uint16_t)rem.y == 0 && iTop[1] + R > 0)
                                bestH.y = max(bestH.y, (int)(mx >> 16) + dr.cost - dr.bias -
                                                           dr.d * (iTop[1] + R - 1 + j));
                        }
                    }
                }
            }
        }
        // The next block reads this block's row-buffer entries from the
        // same lane: order the stores before those loads.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }

    __device__ __forceinline__ static bool wellFormed(const FwdArgs &a, const WorkItem &w)
    {
        // A malformed descriptor is skipped rather than allowed to run past
        // the row buffer or loop without bound.
        return !(w.count < 1 || w.count > 128 || w.maxN < 1 || rowColsFor(w.maxN) > a.rowCols || w.nblocks < 1 ||
                 w.nblocks > (1 << 20) / R + 1);
    }

    __device__ __forceinline__ static void run(const FwdArgs &a)
    {
        __shared__ uint32_t sProf[16];
        __shared__ int16_t sT[33 * 33];
        // Under drift t = s - o + drift for real codes, 0 for the padding code.
        if constexpr (DNA) {
            if (threadIdx.x < 16) {
                uint32_t w = a.dnaProfile[threadIdx.x];
                if (!LOC && (int)(threadIdx.x & 7) < a.alpha)
                    w += (uint32_t)a.drift.d * (0x01010101u >> (32 - 8 * min(a.alpha, 4)));
                sProf[threadIdx.x] = w;
            }
        } else {
            const int TW = a.alpha + 1;
            for (int i = threadIdx.x; i < TW * TW; i += blockDim.x) {
                const bool pad = i / TW == a.alpha || i % TW == a.alpha;
                sT[i] = LOC ? a.tTable[i] : pad ? (int16_t)0 : (int16_t)(a.tTable[i] + a.drift.d);
            }
        }
        __syncthreads();

        const int lane = threadIdx.x & 63;
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const size_t slot = (size_t)blockIdx.x * (blockDim.x >> 6) + wave;
        uint2 *rb = reinterpret_cast<uint2 *>(a.rowbuf) + slot * (size_t)a.rowCols * 64 + lane;
        for (;;) {
            // Branch-free: every lane takes part (lane 0 adds 1), so no
            // lane-0 branch can be merged with another around the back edge
            // and this readfirstlane always runs with lane 0 active.
            int it = (int)atomicAdd(a.queue, lane == 0 ? 1u : 0u);
            it = __builtin_amdgcn_readfirstlane(it);
            if (it >= a.nItems)
                break;
            const WorkItem w = a.items[it];
            const bool ok = wellFormed(a, w);
            Couple c;
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int sidx = 2 * lane + x;
                const int pid = (ok && sidx < w.count) ? a.order[w.first + sidx] : -1;
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
                c.p[x] = w.nblocks * R - 1 - m;
            }
            s16x2 best = splat(a.gapOpen);                  // local: G of the best cell
            int2 bestH = make_int2(INT32_MIN, INT32_MIN);   // global modes: H
            const int nb = ok ? w.nblocks : 0;
            const bool topFree = !(TRK & kTrackLocal) && (a.mode & SQMI_FREE_TOP) != 0;
            if (nb > 0) {
                if (topFree)
                    block<true, true>(a, c, 0, w.maxN, nb == 1, rb, sProf, sT, best, bestH);
                else
                    block<true, false>(a, c, 0, w.maxN, nb == 1, rb, sProf, sT, best, bestH);
            }
            for (int b = 1; b < nb; ++b)
                block<false, false>(a, c, b, w.maxN, b == nb - 1, rb, sProf, sT, best, bestH);
            if constexpr (LOC)
                bestH = make_int2((int)best.x - a.gapOpen, (int)best.y - a.gapOpen);
            if (c.pid[0] >= 0)
                a.scores[c.pid[0]] = bestH.x;
            if (c.pid[1] >= 0)
                a.scores[c.pid[1]] = bestH.y;
        }
    }
};

// Register budgets: four waves per SIMD (128 VGPRs) for 16 rows per lane, three
// for local alignment (its running maximum and padding masks), two for 32 rows.
// What the compiler spills there (up to 108 registers) belongs to the blocks'
// set-up, but for a free first row's block, whose column loop reads some back.
template <int R, uint32_t TRK>
constexpr int laneWaves() { return R >= 32 ? 2 : (TRK & kTrackLocal) ? 3 : 4; }

template <int R, bool DNA, uint32_t TRK>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(laneWaves<R, TRK>()))) void kLane16(FwdArgs a)
{
    Lane16<R, DNA, TRK>::run(a);
}

template <int R, bool DNA>
const void *laneKernel(const Variant16 &v)
{
#define SQMI_TRK(t)                                                                                        \
    case t:                                                                                                \
        return v.wide ? (const void *)&kLane16<R, DNA, (t) | kWideVals> : (const void *)&kLane16<R, DNA, (t)>;
    switch (v.track) {
        SQMI_TRK(kTrackEnd)
        SQMI_TRK(kTrackBottom)
        SQMI_TRK(kTrackRight)
        SQMI_TRK(kTrackBottom | kTrackRight)
        case kTrackLocal: return (const void *)&kLane16<R, DNA, kTrackLocal>;
        default: return nullptr;
    }
#undef SQMI_TRK
}

const void *laneKernelFor(const Variant16 &v)
{
    if (v.G != 1)
        return nullptr;
    if (v.R == 16)
        return v.dna ? laneKernel<16, true>(v) : laneKernel<16, false>(v);
    if (v.R == 32)
        return v.dna ? laneKernel<32, true>(v) : laneKernel<32, false>(v);
    return nullptr;
}

}  // namespace

bool laneSupported(const Variant16 &v) { return laneKernelFor(v) != nullptr; }

int laneRowCols(int maxN, int R)
{
    return R >= 32 ? Lane16<32, true, kTrackEnd>::rowColsFor(maxN) : Lane16<16, true, kTrackEnd>::rowColsFor(maxN);
}

int occupancyLane16(const Variant16 &v)
{
    const void *k = laneKernelFor(v);
    if (!k)
        return 0;
    int blocks = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k, 256, 0) != hipSuccess)
        return 1;
    return blocks > 0 ? blocks : 1;
}

hipError_t launchLane16(const Variant16 &v, const FwdArgs &args, int gridBlocks, hipStream_t stream)
{
    const void *k = laneKernelFor(v);
    if (!k)
        return hipErrorInvalidValue;
    FwdArgs copy = args;
    void *params[] = {&copy};
    return hipLaunchKernel(k, dim3(gridBlocks), dim3(256), params, 0, stream);
}

}  // namespace sqmi
