// kernels.hip -- gfx950 kernels of the batched affine-gap alignment engine
// other than the packed kernels (score16.hpp, trace16.hpp): the int32 per-pair sweep, the
// traceback walks and count kernels, the fills; and the dispatch to the
// packed kernels' instantiation units (score16.hip, trace16.hip).
#include <algorithm>
#include <type_traits>

#include "kernels.hpp"
#include "packed16.hpp"
#include "band16_parts.hpp"
#include "score16_parts.hpp"
#include "seqan_amd.h"

namespace sqmi {
namespace {
// ---------------------------------------------------------------------------
// int32, one thread per pair: the textbook column sweep with the reference's
// border and tracking rules.  Used for pairs whose values could leave the
// int16 window.
// ---------------------------------------------------------------------------
constexpr int kNeg32 = INT32_MIN / 2;   // DPCellDefaultInfinity (dp_cell.h:141-146)

__device__ __forceinline__ bool tracked32(uint32_t mode, int col, int cell)
{
    if (mode & SQMI_LOCAL)
        return true;
    if (cell == 2)
        return col == 2 || (mode & SQMI_FREE_BOTTOM);
    return col == 2 && (mode & SQMI_FREE_RIGHT);
}

__global__ __launch_bounds__(256) void kSimple32(Simple32Args a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.nIds)
        return;
    const int pid = a.ids[t];
    const int64_t ho = a.hOff[pid], vo = a.vOff[pid];
    const int64_t n = a.hOff[pid + 1] - ho, m = a.vOff[pid + 1] - vo;
    const uint8_t *h = a.hRes + ho;
    const uint8_t *v = a.vRes + vo;
    int32_t *H = a.scratch + 2 * a.scratchOff[t];
    int32_t *E = H + (m + 1);
    const int32_t o = a.gapOpen, e = a.gapExtend;
    const uint32_t mode = a.mode;
    const bool local = (mode & SQMI_LOCAL) != 0;
    const int A = a.alpha;
    int32_t best = kNeg32;
    {
        int32_t F = kNeg32;
        H[0] = 0;
        E[0] = kNeg32;
        if (tracked32(mode, 0, 0) && H[0] > best)
            best = H[0];
        for (int64_t i = 1; i <= m; ++i) {
            if (local || (mode & SQMI_FREE_LEFT)) {
                H[i] = 0;
            } else {
                F = max(F + e, H[i - 1] + o);
                H[i] = F;
            }
            E[i] = kNeg32;
            if (tracked32(mode, 0, i == m ? 2 : 1) && H[i] > best)
                best = H[i];
        }
    }
    for (int64_t j = 1; j <= n; ++j) {
        const int col = (j == n) ? 2 : 1;
        const int hj = min((int)h[j - 1], A - 1);
        const int32_t *row = a.table + hj * A;
        int32_t diag = H[0];
        int32_t F = kNeg32;
        if (local || (mode & SQMI_FREE_TOP)) {
            H[0] = 0;
        } else {
            E[0] = max(E[0] + e, H[0] + o);
            H[0] = E[0];
        }
        if (tracked32(mode, col, 0) && H[0] > best)
            best = H[0];
        int32_t up = H[0];
        for (int64_t i = 1; i <= m; ++i) {
            const int32_t d = diag + row[min((int)v[i - 1], A - 1)];
            diag = H[i];
            const int32_t ei = max(E[i] + e, H[i] + o);
            E[i] = ei;
            F = max(F + e, up + o);
            int32_t x = max(d, max(F, ei));
            if (local)
                x = max(x, 0);
            H[i] = x;
            up = x;
            if (tracked32(mode, col, i == m ? 2 : 1) && x > best)
                best = x;
        }
    }
    a.scores[pid] = best;
}

__global__ void kFillScores(int32_t *scores, const int32_t *ids, int n, int32_t value)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n)
        scores[ids[t]] = value;
}

__global__ void kFill32(uint32_t *p, size_t n, uint32_t value)
{
    // 16 bytes a thread from the first 16-byte boundary on.
    const size_t head = min(n, (size_t)((16 - (reinterpret_cast<uintptr_t>(p) & 15)) & 15) / 4);
    const size_t quads = (n - head) / 4, t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint4 *q = reinterpret_cast<uint4 *>(p + head);
    for (size_t t = t0; t < quads; t += (size_t)gridDim.x * blockDim.x)
        q[t] = make_uint4(value, value, value, value);
    if (t0 < head)
        p[t0] = value;
    if (t0 < n - head - 4 * quads)
        p[head + 4 * quads + t0] = value;
}

// Exclusive prefix sums of the row lengths (one workgroup of 1024 threads:
// thread t sums a contiguous chunk, the chunk sums are scanned in LDS, and
// each thread writes its chunk's prefixes).  start[n] is the total.
__global__ __launch_bounds__(1024) void kScanLengths(const int64_t *len, int64_t *start, int64_t n)
{
    __shared__ int64_t part[1024];
    const int t = threadIdx.x;
    const int64_t chunk = (n + 1023) / 1024, b = min(n, t * chunk), e = min(n, b + chunk);
    int64_t sum = 0;
    for (int64_t i = b; i < e; ++i)
        sum += len[i];
    part[t] = sum;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const int64_t add = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += add;
        __syncthreads();
    }
    int64_t run = part[t] - sum;
    for (int64_t i = b; i < e; ++i) {
        start[i] = run;
        run += len[i];
    }
    if (t == 1023)
        start[n] = part[1023];
}

// Rows from the ends of their segments (row i ends at src + off[i + 1]) to
// dst + off[0] + start[i], back to back: one wavefront per row.
__global__ __launch_bounds__(256) void kPackRows(const uint8_t *src, const int64_t *off, const int64_t *len,
                                                 const int64_t *start, uint8_t *dst, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= n)
        return;
    const int64_t L = len[i];
    const uint8_t *s = src + off[i + 1] - L;
    uint8_t *d = dst + off[0] + start[i];
    for (int64_t k = threadIdx.x & 63; k < L; k += 64)
        d[k] = s[k];
}

// ---------------------------------------------------------------------------
// Traceback.  The walk follows _computeTraceback / _doTracebackGoDiagonal /
// _doTracebackGoVertical / _doTracebackGoHorizontal (dp_traceback_impl.h:
// 115-546) over trace bits with the encoding of the trace records (bit 0: E
// opened, 1: F opened, 2: not diagonal, 3: E beats F), and counts the
// alignment the way computeAlignmentStats reads its rows
// (evaluate_alignment.h:215-300): one substitution count per aligned pair
// (index h * alpha + v), and per maximal run of gaps in one row one open and
// run-1 extensions.  A run is maximal in either reading direction, so the
// counts can be taken while walking backwards.
//
// With gap open == gap extend the reference runs its linear-gap algorithm
// (_usesAffineGaps, dp_setup.h:244-260; dp_formula_linear.h:62-106).  Its
// cells hold the same values and the same own direction (diagonal wins ties,
// then vertical), which the trace bits record; but it keeps no gap matrices,
// so every gap step re-reads the direction of the cell it reaches, and the
// end cell is taken as it is (no _correctTraceValue for linear gaps,
// dp_algorithm_impl.h:1180-1188).
// ---------------------------------------------------------------------------
constexpr uint32_t kBitEOpen = 1, kBitFOpen = 2, kBitNotDiag = 4, kBitHori = 8;
// Local alignment (byte trace only): the cell did not beat 0, so its trace
// value is NONE and a walk that reaches it stops there.
constexpr uint32_t kBitStop = 16;

__device__ __forceinline__ int dirOf(uint32_t bits)   // 0 diagonal, 1 vertical, 2 horizontal
{
    return (bits & kBitNotDiag) ? ((bits & kBitHori) ? 2 : 1) : 0;
}

template <class Bits>
__device__ __forceinline__ void walkCounts(int n, int m, const uint8_t *h, const uint8_t *v, int A, int score, int endE,
                                           int endF, Bits &bits, int32_t *cnt, uint8_t *opEnd = nullptr,
                                           int64_t *opLen = nullptr, int i0 = -1, int j0 = -1,
                                           bool local = false, int64_t *begins = nullptr, bool linear = false,
                                           const int32_t *lTab = nullptr, int go = 0, int ge = 0)
{
    // Local walks over packed trace records (lTab given) carry no stop bit:
    // they track H along the path instead (the score at the end cell, minus
    // each diagonal's substitution score, minus gapOpen or gapExtend per gap
    // character by the record's open bit) and stop on the first cell where
    // it is 0, which is where the reference's trace value is NONE.
    int cur = score;
    // The walk starts at the end cell (i0, j0), (m, n) unless free end gaps
    // or a local alignment moved it; in global modes the cells after it are
    // trailing gaps of the rows.  A local walk stops at the first cell whose
    // trace value is NONE (kBitStop) and emits neither trailing nor leading
    // gaps (TraceTail_ / TraceHead_, dp_profile.h:482-492).
    int i = i0 < 0 ? m : i0, j = j0 < 0 ? n : j0;
    if (local) {
        m = i;
        n = j;
    }
    int prev = 0;   // last emitted operation: 0 none / aligned pair, 1 gap in H (vertical), 2 gap in V
    int opens = 0, exts = 0;
    // Rows: one byte per alignment column, written backwards from opEnd
    // ('M' both residues, 'V' gap in the H row, 'H' gap in the V row).
    int64_t nOps = 0;
    auto emit = [&](uint8_t op) {
        if (opEnd)
            opEnd[-1 - nOps] = op;
        ++nOps;
    };
    // Trailing gaps after the end cell: the rest of V, then of H.
    for (int k = i; k < m; ++k) {
        if (prev == 1) ++exts; else ++opens;
        prev = 1;
        emit('V');
    }
    for (int k = j; k < n; ++k) {
        if (prev == 2) ++exts; else ++opens;
        prev = 2;
        emit('H');
    }
    // End cell: F, then E, win ties against the recorded direction
    // (_correctTraceValue, dp_algorithm_impl.h:1190-1207), and a gap start
    // there follows the gap matrix (PreferGapsAtEnd_, dp_traceback_impl.h:115-122).
    int dir;
    bool walk = true;
    {
        const uint32_t b0 = (i > 0 && j > 0) ? bits(i, j) : kBitStop;
        dir = linear ? dirOf(b0) : (endF == score) ? 1 : (endE == score) ? 2 : dirOf(b0);
        if (local && (lTab ? cur <= 0 : (b0 & kBitStop) != 0))
            walk = false;
    }
    while (walk && i > 0 && j > 0) {
        if (dir == 0) {
            const int hc = min((int)h[j - 1], A - 1), vc = min((int)v[i - 1], A - 1);
            cnt[hc * A + vc] += 1;
            if (lTab)
                cur -= lTab[hc * A + vc];
            emit('M');
            prev = 0;
            --i;
            --j;
        } else if (dir == 1) {
            for (;;) {
                const bool open = (bits(i, j) & kBitFOpen) != 0;
                if (prev == 1) ++exts; else ++opens;
                prev = 1;
                cur -= (open || linear) ? go : ge;
                emit('V');
                const bool stop = linear || open || i == 1;
                --i;
                if (stop)
                    break;
            }
        } else {
            for (;;) {
                const bool open = (bits(i, j) & kBitEOpen) != 0;
                if (prev == 2) ++exts; else ++opens;
                prev = 2;
                cur -= (open || linear) ? go : ge;
                emit('H');
                const bool stop = linear || open || j == 1;
                --j;
                if (stop)
                    break;
            }
        }
        if (i > 0 && j > 0) {
            if (local && lTab && cur == 0)
                break;
            const uint32_t b = bits(i, j);
            dir = dirOf(b);
            if (local && !lTab && (b & kBitStop))
                break;
        }
    }
    if (local) {
        // The window starts where the walk stopped (dp_traceback_adaptor.h:
        // 87-93); an empty window keeps both begins at 0.
        if (begins && nOps > 0) {
            begins[0] = j;
            begins[1] = i;
        }
        i = j = 0;
    }
    // Leading gaps down to the origin: first the column, then the row
    // (dp_traceback_impl.h:522-545).
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
    if (opLen)
        *opLen = nOps;
}

// The same walk by a group of 16 lanes per pair: the lanes read the bits of
// the next 16 cells of the diagonal (or of the gap) at once, so a walk waits
// for memory once per run of equal moves (or per 16 of them) instead of once
// per move.  What bounds it then is the records' traffic: each cell's record
// sits in a line of its own (65,536 pairs of 1 kbp 1.85 -> 1.39 ms; 8,191
// uneven pairs of up to 10 kbp, where the longest walk counts, 13.8 -> 0.5 ms;
// 8,192 protein pairs local 1.24 -> 0.1 ms; 65,536 banded pairs of 150 bp
// 0.67 -> 0.17 ms).  The state is kept alike in all lanes of the group;
// groups of a wave diverge as they like (a group's lanes never do, outside
// predicated statements).
//
// W lanes per pair: 16, or a whole wave (64) in calls of few pairs, which wait
// for their longest walk (kWalkWavePairs).
constexpr int kWalkLanes = 16;

template <int W>
__device__ __forceinline__ uint64_t groupBallot(bool p)
{
    return W == 64 ? __ballot(p) : (__ballot(p) >> (threadIdx.x & 48)) & 0xffffu;
}

struct WalkEnd {
    int score, i, j, e, f;   // the end cell
};

template <int W, class Bits>
__device__ __forceinline__ void walkGroup(int n, int m, const uint8_t *h, const uint8_t *v, int A, const WalkEnd &end,
                                          const Bits &bits, int32_t *cnt, uint8_t *opEnd, int64_t *opLen, bool local,
                                          int64_t *begins, bool linear, bool alwaysOpen, const int32_t *lTab, int go,
                                          int ge)
{
    const int t = threadIdx.x & (W - 1);
    int cur = end.score, i = end.i, j = end.j;
    if (local) {
        m = i;
        n = j;
    }
    int prev = 0, opens = 0, exts = 0;
    int64_t nOps = 0;
    // A run of k equal moves: 0 aligned pairs, 1 gap in H ('V'), 2 gap in V.
    auto emit = [&](int kind, int k) {
        if (kind > 0 && k > 0) {
            opens += prev == kind ? 0 : 1;
            exts += prev == kind ? k : k - 1;
        }
        if (k > 0)
            prev = kind;
        if (opEnd)
            for (int q = t; q < k; q += W)
                opEnd[-1 - nOps - q] = kind == 0 ? 'M' : kind == 1 ? 'V' : 'H';
        nOps += k;
    };
    emit(1, m - i);   // trailing gaps after the end cell
    emit(2, n - j);
    bool walk = i > 0 && j > 0, first = true;
    int known = -1;   // direction of (i, j) by the end-cell rule
    if (walk) {
        const uint32_t b0 = bits(i, j);
        known = linear ? dirOf(b0) : end.f == end.score ? 1 : end.e == end.score ? 2 : dirOf(b0);
        if (local && (lTab ? cur <= 0 : (b0 & kBitStop) != 0))
            walk = false;
    }
    while (walk) {
        // Aligned pairs from (i, j) up the diagonal.
        const int ii = i - t, jj = j - t;
        const bool valid = ii > 0 && jj > 0;
        // The residues with the bits, though cells past the run do not need
        // them: one wait instead of two.
        const int rh = valid ? h[jj - 1] : 0, rw = valid ? v[ii - 1] : 0;
        const uint32_t b = valid ? bits(ii, jj) : 0;
        int d = valid ? dirOf(b) : 3;
        if (t == 0 && first)
            d = known;
        const bool none = local && !lTab && (b & kBitStop) != 0 && !(first && t == 0);
        const uint64_t stops = groupBallot<W>(d != 0 || none);
        int r = stops ? __builtin_ctzll(stops) : W;
        bool stopped = false;
        const int hv = min(rh, A - 1) * A + min(rw, A - 1);
        if (lTab) {
            // H along the run; the walk stops on the first cell where it is 0.
            int sum = t < r ? lTab[hv] : 0;
#pragma unroll
            for (int q = 1; q < W; q <<= 1) {
                const int o = __shfl_up(sum, q, W);
                sum += t >= q ? o : 0;
            }
            const uint64_t zero = groupBallot<W>(t < r && cur == sum && ii > 1 && jj > 1);
            if (zero) {
                r = __builtin_ctzll(zero) + 1;
                stopped = true;
            }
            if (r > 0)
                cur -= __shfl(sum, r - 1, W);
        }
        if (t < r)
            atomicAdd(cnt + hv, 1);
        emit(0, r);
        i -= r;
        j -= r;
        if (stopped || i <= 0 || j <= 0)
            break;
        if (r == W) {
            first = false;
            continue;
        }
        if (__shfl((int)none, r, W))
            break;
        const bool vert = __shfl(d, r, W) == 1;
        first = false;
        // A gap: up to the cell that opened it, or row / column 1.
        for (;;) {
            const int gi = vert ? i - t : i, gj = vert ? j : j - t, at = vert ? gi : gj;
            const uint32_t gb = at > 0 ? bits(gi, gj) : 0;
            const bool open = alwaysOpen || (gb & (vert ? kBitFOpen : kBitEOpen)) != 0;
            const uint64_t gEnd = groupBallot<W>(at > 0 && (linear || open || at == 1));
            const int g = gEnd ? __builtin_ctzll(gEnd) + 1 : W;
            const bool opened = linear || __shfl((int)open, g - 1, W) != 0;
            emit(vert ? 1 : 2, g);
            cur -= ge * (g - 1) + (gEnd && opened ? go : ge);
            if (vert)
                i -= g;
            else
                j -= g;
            if (gEnd)
                break;
        }
        if (i <= 0 || j <= 0 || (lTab && cur == 0))
            break;
    }
    if (local) {
        // The window starts where the walk stopped (dp_traceback_adaptor.h:
        // 87-93); an empty window keeps both begins at 0.
        if (begins && nOps > 0 && t == 0) {
            begins[0] = j;
            begins[1] = i;
        }
        i = j = 0;
    }
    // Leading gaps down to the origin: first the column, then the row
    // (dp_traceback_impl.h:522-545).
    emit(1, i);
    emit(2, j);
    if (t == 0) {
        atomicAdd(cnt + A * A, opens);
        atomicAdd(cnt + A * A + 1, exts);
        if (opLen)
            *opLen = nOps;
    }
}

// Trace bits of cell (i, j) of one pair from the packed records of kTrace16.
struct Bits16 {
    const uint4 *trace;
    TraceLoc loc;
    __device__ __forceinline__ uint32_t operator()(int i, int j) const
    {
        const int r = loc.p + i;
        const int b = r / kTraceRows, rr = r % kTraceRows;
        if (loc.lanes == 64) {
            const int l = rr / 4, sh = rr % 4 + 8 * loc.half;
            const uint32_t w = reinterpret_cast<const uint32_t *>(trace + loc.rec0 * 64)[((int64_t)b * loc.steps + (j + l)) * 64 + l];
            return ((w >> sh) & 1u) | (((w >> (sh + 16)) & 1u) << 1) | (((w >> (sh + 4)) & 1u) << 2) |
                   (((w >> (sh + 20)) & 1u) << 3);
        }
        const int l = rr / 16, k = rr % 16;
        const uint4 w = trace[(loc.rec0 + (int64_t)b * loc.steps + (j + l)) * 64 + loc.lane0 + l];
        const uint32_t ef = k < 8 ? w.x : w.y, dx = k < 8 ? w.z : w.w;
        const int sh = (k & 7) + 8 * loc.half;
        return ((ef >> sh) & 1u) | (((ef >> (sh + 16)) & 1u) << 1) | (((dx >> sh) & 1u) << 2) |
               (((dx >> (sh + 16)) & 1u) << 3);
    }
};

// Trace bytes of a banded pair (kBandedTrace): row i - 1, lane j - i - lo.
struct BandBits {
    const uint8_t *trace;
    int S;
    int lo;
    int w;   // diagonals of the clipped band (<= S)
    int n;
    __device__ __forceinline__ uint32_t operator()(int i, int j) const
    {
        // An optimal path stays inside the band (cells outside are -inf).
        // Cells outside the clipped band or past column n read as a stop,
        // so that no walk can step onto trace bytes the trace kernel did
        // not write (the lanes of a segment beyond the band's width).
        const int c = j - i - lo;
        if (c < 0 || c >= w || j > n)
            return kBitStop;
        return trace[(int64_t)(i - 1) * S + c];
    }
};

// Threads of a walk workgroup: counts accumulate in LDS (alpha^2 + 2 words per
// pair, at most 1,026), so large alphabets take fewer pairs per workgroup.
int walkThreads(int alpha) { return alpha <= 7 ? 256 : 64; }

__global__ __launch_bounds__(256) void kBandedWalk(BandedWalkArgs a)
{
    extern __shared__ int32_t sCnt[];
    const int A = a.alpha, S = A * A + 2;
    const int t = threadIdx.x & (kWalkLanes - 1), q = threadIdx.x / kWalkLanes;
    const int id = blockIdx.x * (blockDim.x / kWalkLanes) + q;
    int32_t *cnt = sCnt + q * S;
    for (int k = t; k < S; k += kWalkLanes)
        cnt[k] = 0;
    __syncthreads();
    if (id < a.nIds) {
        const int pid = a.ids[id];
        const int64_t ho = a.hOff[pid], vo = a.vOff[pid];
        const int n = (int)(a.hOff[pid + 1] - ho), m = (int)(a.vOff[pid + 1] - vo);
        const int lo = (int)(a.lower > -(int64_t)m ? a.lower : -(int64_t)m);   // the band clipped to the matrix
        const int up = (int)(a.upper < (int64_t)n ? a.upper : (int64_t)n);
        const BandBits bits{a.trace + a.traceOff[id], a.segLanes, lo, min(up - lo + 1, a.segLanes), n};
        const WalkEnd end{a.scores[pid], a.endIJ[2 * pid], a.endIJ[2 * pid + 1], a.endEF[2 * pid], a.endEF[2 * pid + 1]};
        walkGroup<kWalkLanes>(n, m, a.hRes + ho, a.vRes + vo, A, end, bits, cnt,
                              a.ops ? a.ops + a.opOff[pid + 1] : nullptr, a.ops ? a.opLen + pid : nullptr, a.local != 0,
                              a.begins ? a.begins + 2 * pid : nullptr, a.linear != 0, false, nullptr, 0, 0);
    }
    __syncthreads();
    if (id < a.nIds) {
        int32_t *out = a.counts + (int64_t)a.ids[id] * S;
        for (int k = t; k < S; k += kWalkLanes)
            out[k] = cnt[k];
    }
}

template <int W>
__global__ __launch_bounds__(256) void kWalk16(WalkArgs a)
{
    extern __shared__ int32_t sCnt[];
    const int A = a.alpha, S = A * A + 2;
    const int t = threadIdx.x & (W - 1), q = threadIdx.x / W;
    const int id = blockIdx.x * (blockDim.x / W) + q;
    int32_t *cnt = sCnt + q * S;
    for (int k = t; k < S; k += W)
        cnt[k] = 0;
    __syncthreads();
    if (id < a.nPairs) {
        const int pid = a.ids[id];
        const TraceLoc loc = a.locs[id];
        const int64_t ho = a.hOff[pid], vo = a.vOff[pid];
        const int n = (int)(a.hOff[pid + 1] - ho), m = (int)(a.vOff[pid + 1] - vo);
        // The end cell.  Local: the candidates' first strict maximum in
        // column order.  Global: the last unit's bottom-row candidate, unless
        // a cell of column n beats it (rows ascend with the units).
        WalkEnd end{INT32_MIN, 0x7fffffff, 0x7fffffff, INT32_MIN, INT32_MIN};
        for (int k = t; k < loc.nEnds; k += W) {
            const TraceEnd c = a.ends[loc.end0 + (int64_t)k * loc.endStride];
            const bool take = a.local ? c.v > end.score || (c.v == end.score && (c.j < end.j || (c.j == end.j && c.i < end.i)))
                                      : c.rv > end.score || (c.rv == end.score && c.ri < end.i);
            if (take)
                end = a.local ? WalkEnd{c.v, c.i, c.j, c.e, c.f} : WalkEnd{c.rv, c.ri, c.rj, c.re, c.rf};
        }
#pragma unroll
        for (int d = 1; d < W; d <<= 1) {
            const WalkEnd o{__shfl_xor(end.score, d, W), __shfl_xor(end.i, d, W),
                            __shfl_xor(end.j, d, W), __shfl_xor(end.e, d, W),
                            __shfl_xor(end.f, d, W)};
            if (o.score > end.score || (o.score == end.score && (o.j < end.j || (o.j == end.j && o.i < end.i))))
                end = o;
        }
        if (a.local) {
            if (end.j == 0x7fffffff)   // no cell above 0: an empty window
                end = WalkEnd{0, 0, 0, INT32_MIN, INT32_MIN};
        } else {
            const TraceEnd c = a.ends[loc.end0 + (int64_t)(loc.nEnds - 1) * loc.endStride];
            if (c.v != INT32_MIN && c.v >= end.score)
                end = WalkEnd{c.v, c.i, c.j, c.e, c.f};
        }
        if (t == 0)
            a.scores[pid] = end.score;
        const Bits16 bits{a.trace, loc};
        walkGroup<W>(n, m, a.hRes + ho, a.vRes + vo, A, end, bits, cnt, a.ops ? a.ops + a.opOff[pid + 1] : nullptr,
                  a.ops ? a.opLen + pid : nullptr, a.local != 0, a.begins ? a.begins + 2 * pid : nullptr,
                  a.linear != 0, a.gapExtend < a.gapOpen, a.local ? a.table : nullptr, a.gapOpen, a.gapExtend);
    }
    __syncthreads();
    if (id < a.nPairs) {
        int32_t *out = a.counts + (int64_t)a.ids[id] * S;
        for (int k = t; k < S; k += W)
            out[k] = cnt[k];
    }
}

// int32 forward with trace bytes (same encoding), column-major with column
// stride m + 1, followed by the same walk.  For pairs outside the int16 window.
__global__ __launch_bounds__(256) void kCounts32(Counts32Args a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.nIds)
        return;
    const int pid = a.ids[t];
    const int A = a.alpha, S = A * A + 2;
    const int64_t ho = a.hOff[pid], vo = a.vOff[pid];
    const int n = (int)(a.hOff[pid + 1] - ho), m = (int)(a.vOff[pid + 1] - vo);
    const uint8_t *h = a.hRes + ho;
    const uint8_t *v = a.vRes + vo;
    uint8_t *base = a.scratch + a.scratchOff[t];
    int32_t *H = reinterpret_cast<int32_t *>(base);
    int32_t *E = H + (m + 1);
    uint8_t *T = base + 8 * (int64_t)(m + 1);
    const int64_t CS = m + 1;
    const int32_t o = a.gapOpen, e = a.gapExtend;
    int32_t *cnt = a.counts + (int64_t)pid * S;
    for (int k = 0; k < S; ++k)
        cnt[k] = 0;
    // Free end gaps (AlignConfig, dp_setup.h:57-182): a free first row /
    // column is 0; the result is the first strict maximum over the tracked
    // cells in column order: (m, n), the last row if it is free, the last
    // column if it is free (dp_scout.h:169-210, dp_meta_info.h:178-221).
    // Local: both borders are 0, a cell that does not beat 0 is 0 with trace
    // NONE (dp_formula_affine.h:110-118), and every cell is tracked
    // (dp_scout_simd.h:427-440).
    const bool local = (a.mode & SQMI_LOCAL) != 0;
    const bool freeTop = local || (a.mode & SQMI_FREE_TOP) != 0, freeLeft = local || (a.mode & SQMI_FREE_LEFT) != 0;
    const bool freeRight = local || (a.mode & SQMI_FREE_RIGHT) != 0;
    const bool freeBottom = local || (a.mode & SQMI_FREE_BOTTOM) != 0;
    // Banded (globalAlignment / localAlignment with lowerDiag, upperDiag,
    // global_alignment_banded.h:152-181, local_alignment_banded.h:242-259):
    // column j holds rows [j - upper, j - lower] only; the rest are -inf,
    // which is what the reference's band-edge recursions give
    // (dp_formula_affine.h:129-230).  Rows below the band keep the -inf
    // they start with; rows above it are never read again.
    const bool banded = a.banded != 0;
    const int64_t lo = a.lower, hi = a.upper;
    int32_t best = kNeg32, bestE = kNeg32, bestF = kNeg32;
    int bi = m, bj = n;
    auto track = [&](bool lastCol, int i, int j, int32_t hv, int32_t ev, int32_t fv) {
        const bool tracked = local || ((i == m) ? (lastCol || freeBottom) : (lastCol && freeRight));
        if (tracked && hv > best) {
            best = hv;
            bestE = ev;
            bestF = fv;
            bi = i;
            bj = j;
        }
    };
    {
        int32_t F = kNeg32;
        H[0] = (banded && (lo > 0 || hi < 0)) ? kNeg32 : 0;
        E[0] = kNeg32;
        for (int i = 1; i <= m; ++i) {
            if (banded && (-i < lo || -i > hi)) {
                H[i] = kNeg32;
                E[i] = kNeg32;
                F = kNeg32;
                continue;
            }
            if (freeLeft) {
                H[i] = 0;
            } else {
                F = max(F + e, H[i - 1] + o);
                H[i] = F;
            }
            E[i] = kNeg32;
            track(false, i, 0, H[i], E[i], freeLeft ? kNeg32 : F);
        }
    }
    for (int j = 1; j <= n; ++j) {
        const int hj = min((int)h[j - 1], A - 1);
        const int32_t *row = a.table + hj * A;
        int32_t diag = H[0];
        int32_t F = kNeg32;
        if (banded && (j < lo || j > hi)) {
            H[0] = kNeg32;
            E[0] = kNeg32;
        } else if (freeTop) {
            H[0] = 0;
        } else {
            E[0] = max(E[0] + e, H[0] + o);
            H[0] = E[0];
        }
        track(j == n, 0, j, H[0], E[0], kNeg32);
        int32_t up = H[0];
        uint8_t *Tc = T + (int64_t)j * CS;
        int i0 = 1, i1 = m;
        if (banded) {
            i0 = (int)max<int64_t>(1, j - hi);
            i1 = (int)min<int64_t>(m, j - lo);
            if (i0 > 1) {
                diag = H[i0 - 1];   // column j - 1's value: (i0 - 1, j - 1) is in the band
                up = kNeg32;
            }
        }
        for (int i = i0; i <= i1; ++i) {
            const int32_t d = diag + row[min((int)v[i - 1], A - 1)];
            diag = H[i];
            const int32_t extE = E[i] + e, opnE = H[i] + o;
            uint32_t tb = extE < opnE ? kBitEOpen : 0u;
            const int32_t ei = max(extE, opnE);
            E[i] = ei;
            const int32_t extF = F + e, opnF = up + o;
            tb |= extF < opnF ? kBitFOpen : 0u;
            F = max(extF, opnF);
            const int32_t fe = F < ei ? ei : F;
            int32_t x = d;
            if (d < fe) {
                x = fe;
                tb |= kBitNotDiag | (F < ei ? kBitHori : 0u);
            }
            if (local && !(0 < x)) {
                x = 0;
                tb = kBitStop;
            }
            Tc[i] = (uint8_t)tb;
            H[i] = x;
            up = x;
            track(j == n, i, j, x, ei, F);
        }
    }
    a.scores[pid] = best;
    // A band whose lower diagonal ends on the last row: the reference tracks
    // that cell from the next column's code path (dp_algorithm_impl.h:
    // 843-862) and its traceback then takes the cell's own direction, with
    // no preference for the vertical gap.
    if (banded && bi == m && (int64_t)bj - bi == lo)
        bestF = kNeg32;
    auto bits = [&](int i, int j) -> uint32_t { return T[(int64_t)j * CS + i]; };
    walkCounts(n, m, h, v, A, best, bestE, bestF, bits, cnt, a.ops ? a.ops + a.opOff[pid + 1] : nullptr,
               a.ops ? a.opLen + pid : nullptr, bi, bj, local, a.begins ? a.begins + 2 * pid : nullptr, o == e);
}

}  // namespace

int wavesPerBlock16() { return 4; }

namespace {

const void *scoreKernel(bool dna, int kind)
{
    switch (kind) {
        case kScoreGlobal: return dna ? scoreDnaGlobal() : scoreTabGlobal();
        case kScoreRight: return dna ? scoreDnaRight() : scoreTabRight();
        case kScoreLocal: return dna ? scoreDnaLocal() : scoreTabLocal();
        default: return nullptr;
    }
}

}  // namespace

int occupancyScore16(bool dna, int kind, int waves)
{
    int blocks = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, scoreKernel(dna, kind), 64 * waves, 0) != hipSuccess)
        return 1;
    return blocks > 0 ? blocks : 1;
}

static const void *bandKernel(const BandVariant &v)
{
    using Part = const void *(*)(int, bool, bool);
    static constexpr Part parts[2][3] = {{bandTabEnd, bandTabFree, bandTabLocal}, {bandDnaEnd, bandDnaFree, bandDnaLocal}};
    return v.kind < 0 || v.kind > 2 ? nullptr : parts[v.dna][v.kind](v.R, v.wide, v.lds);
}

int bandRingCols(int maxN, int64_t lower, int64_t upper, int R)
{
    // The smallest power of two of at least W - 1 + R + 10 columns; when that
    // reaches the pair's whole width the buffer is linear (a power of two
    // no smaller than bandRowCols).
    const int64_t need = std::min<int64_t>(upper - lower + R + 10, (int64_t)bandRowCols(maxN));
    int c = 1;
    while (c < need)
        c <<= 1;
    return c;
}

int bandLdsRingBytes(int bandCols)
{
    // A ring of bandCols columns x 64 lanes x 8 bytes, when it leaves room
    // for the static tables in the 160 KB of LDS per CU.
    const int64_t bytes = (int64_t)64 * bandCols * 8;
    return bytes > 128 * 1024 ? 0 : (int)bytes;
}

int occupancyBand16(const BandVariant &v, int ringLdsBytes)
{
    const void *k = bandKernel(v);
    int blocks = 0;
    if (!k || (v.lds && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, ringLdsBytes) != hipSuccess))
        return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k, 64 * v.waves, (size_t)ringLdsBytes) != hipSuccess)
        return 1;
    return blocks > 0 ? blocks : 1;
}

hipError_t launchBand16(const BandVariant &v, const FwdArgs &args, int gridBlocks, int ringLdsBytes, hipStream_t stream)
{
    const void *k = bandKernel(v);
    if (!k)
        return hipErrorInvalidValue;
    FwdArgs copy = args;
    void *params[] = {&copy};
    return hipLaunchKernel(k, dim3(gridBlocks), dim3(64 * v.waves), params, (size_t)ringLdsBytes, stream);
}

hipError_t launchScore16(bool dna, int kind, const ScoreArgs &args, int gridBlocks, int waves, hipStream_t stream)
{
    const void *k = scoreKernel(dna, kind);
    if (!k)
        return hipErrorInvalidValue;
    ScoreArgs copy = args;
    void *params[] = {&copy};
    return hipLaunchKernel(k, dim3(gridBlocks), dim3(64 * waves), params, 0, stream);
}

hipError_t launchTrace16(bool dna, uint32_t track, const TraceArgs &args, int gridBlocks, hipStream_t stream)
{
    const void *k = dna ? traceDna(track) : traceTab(track);
    if (!k)
        return hipErrorInvalidValue;
    TraceArgs copy = args;
    void *params[] = {&copy};
    return hipLaunchKernel(k, dim3(gridBlocks), dim3(256), params, 0, stream);
}

int occupancyTrace16(bool dna, uint32_t track)
{
    int blocks = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, dna ? traceDna(track) : traceTab(track), 256, 0) !=
        hipSuccess)
        return 1;
    return blocks > 0 ? blocks : 1;
}

// Up to this many pairs (a wave each fills the chip's SIMDs 16 times) the
// longest walk bounds the kernel, and 64 lanes read four times as far at once:
// 8,191 uneven pairs of up to 10 kbp 0.51 ms against 1.08 with 16 lanes, 8,192
// protein pairs local 0.095 / 0.11; 65,536 pairs of 1 kbp, bound by the
// records' traffic, 2.1 / 1.39.
constexpr int kWalkWavePairs = 16384;

hipError_t launchWalk16(const WalkArgs &args, hipStream_t stream)
{
    if (args.nPairs <= 0)
        return hipSuccess;
    const bool wave = args.nPairs <= kWalkWavePairs;
    const int threads = walkThreads(args.alpha), pairs = threads / (wave ? 64 : kWalkLanes);
    const void *k = wave ? (const void *)&kWalk16<64> : (const void *)&kWalk16<kWalkLanes>;
    WalkArgs copy = args;
    void *params[] = {&copy};
    return hipLaunchKernel(k, dim3((args.nPairs + pairs - 1) / pairs), dim3(threads), params,
                           (size_t)pairs * (args.alpha * args.alpha + 2) * sizeof(int32_t), stream);
}

hipError_t launchBandedWalk(const BandedWalkArgs &args, hipStream_t stream)
{
    if (args.nIds <= 0)
        return hipSuccess;
    const int threads = walkThreads(args.alpha), pairs = threads / kWalkLanes;
    hipLaunchKernelGGL(kBandedWalk, dim3((args.nIds + pairs - 1) / pairs), dim3(threads),
                       (size_t)pairs * (args.alpha * args.alpha + 2) * sizeof(int32_t), stream, args);
    return hipGetLastError();
}

hipError_t launchCounts32(const Counts32Args &args, hipStream_t stream)
{
    if (args.nIds <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(kCounts32, dim3((args.nIds + 255) / 256), dim3(256), 0, stream, args);
    return hipGetLastError();
}

hipError_t launchSimple32(const Simple32Args &args, hipStream_t stream)
{
    if (args.nIds <= 0)
        return hipSuccess;
    dim3 grid((args.nIds + 255) / 256), block(256);
    hipLaunchKernelGGL(kSimple32, grid, block, 0, stream, args);
    return hipGetLastError();
}

hipError_t launchFill32(uint32_t *p, size_t n, uint32_t value, hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    const size_t blocks = std::min<size_t>((n + 1023) / 1024, 2048);
    hipLaunchKernelGGL(kFill32, dim3((unsigned)blocks), dim3(256), 0, stream, p, n, value);
    return hipGetLastError();
}

hipError_t launchPackRows(const uint8_t *src, const int64_t *off, const int64_t *len, int64_t *start, uint8_t *dst,
                          int64_t n, hipStream_t stream)
{
    if (n <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(kScanLengths, dim3(1), dim3(1024), 0, stream, len, start, n);
    hipLaunchKernelGGL(kPackRows, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, stream, src, off, len,
                       (const int64_t *)start, dst, n);
    return hipGetLastError();
}

hipError_t launchFillScores(int32_t *scores, const int32_t *ids, int n, int32_t value, hipStream_t stream)
{
    if (n <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(kFillScores, dim3((n + 255) / 256), dim3(256), 0, stream, scores, ids, n, value);
    return hipGetLastError();
}

}  // namespace sqmi
