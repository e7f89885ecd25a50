// engine.cpp -- host side of the C ABI: validation, exact int16/int32
// routing, length bucketing into wavefront work items, launches.
//
// Behaviour mirrors the reference entry points:
//   globalAlignmentScore / localAlignmentScore (ExecutionPolicy<Parallel,Vectorial>)
//     include/seqan/align_parallel/parallel_align_interface.h:100-145, 332-365
// The reference splits the set into chunks of <= 256 pairs for OpenMP threads
// and each chunk into SIMD batches of 8/16 pairs padded to the batch maximum
// (include/seqan/align/dp_align_simd_helper.h:147-221, 277-347).  Here pairs
// are instead grouped by length across the whole set, so that the pairs that
// share a wavefront have nearly the same shape.
#include "kernels.hpp"
#include "seqan_amd.h"

#include <algorithm>
#ifdef _OPENMP
#include <omp.h>
#endif
#include <chrono>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <new>
#include <string>
#include <thread>
#include <vector>

using namespace sqmi;

namespace {

// A bump allocator over caller-free device memory (the no-allocation entry
// point's scratch array): buffers carved from it are never freed.
struct Arena
{
    char *base = nullptr;
    size_t cap = 0, used = 0;
};

struct DevBuf
{
    void *p = nullptr;
    size_t cap = 0;
    Arena *arena = nullptr;   // set: carve from this arena instead of hipMalloc
    // p lies in the context's stage; the buffer's own memory waits here.
    bool view = false;
    void *own = nullptr;
    size_t ownCap = 0;
};

// Every device buffer a context keeps between calls.
struct Buffers
{
    DevBuf hRes, vRes, hOff, vOff, order, items, queue, rowbuf, strips, scores, tTable, dnaProf, ids32, scratchOff32,
        scratch32, table32, emptyIds;
    // Traceback (sqmi_align_counts).
    DevBuf trace, traceOff, locs, ends, endOff, endEF, endIJ, counts;
    // Long pairs (tiled int32 kernels).
    DevBuf longCk, longRows, longPairs, longWalk, longTrace, longBest, longSched;
    // Alignment rows (sqmi_align_rows, sqmi_align_local_rows).
    DevBuf ops, opOff, opLen, begins, opsPacked, opStart;
    // Banded scores (sqmi_align_score_banded).
    DevBuf bandIds, bandScratch;

    template <class F>
    void forEach(F f)
    {
        for (DevBuf *b : {&hRes, &vRes, &hOff, &vOff, &order, &items, &queue, &rowbuf, &strips, &scores, &tTable, &dnaProf,
                          &ids32, &scratchOff32, &scratch32, &table32, &emptyIds, &trace, &traceOff, &locs, &ends, &endOff, &endEF,
                          &endIJ, &counts, &longCk, &longRows, &longPairs, &longWalk, &longTrace, &longBest, &longSched, &ops, &opOff, &opLen,
                          &begins, &opsPacked, &opStart, &bandIds, &bandScratch})
            f(*b);
    }
};

}  // namespace

namespace {
struct Planned;
}

struct sqmi_context
{
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t ownStream = nullptr;
    int numCUs = 0;
    int64_t l2PerCU = 0;    // bytes of L2 per CU (one L2 per XCD of 32 CUs on gfx950)
    int64_t totalMem = 0;   // device memory, bytes
    std::string lastError;
    sqmi_stats stats{};
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // Long-pair forward: side streams (default priority) that sweep groups
    // of pair couples concurrently, with fork / join events.
    static constexpr int kMaxLongStreams = 4;
    hipStream_t longStreams[kMaxLongStreams] = {};
    hipEvent_t longFork = nullptr, longJoin[kMaxLongStreams] = {};
    Buffers b;
    // A call's offsets, tables and work lists go through pinned memory to
    // one device buffer (stageBegin, put, stageFlush).
    DevBuf stage;
    char *pin = nullptr;
    size_t pinCap = 0, pinUsed = 0, pinSent = 0;
    bool pinOn = false;      // the running call stages its uploads
    struct Down {
        void *dst;
        const void *src;
        size_t bytes;
    };
    std::vector<Down> down;  // results on their way through `pin` (fetch, deliver)
    size_t downUsed = 0, downCap = 0;
    bool pinBusy = false;    // copies from `pin` may be in flight
    Planned *planned = nullptr;   // the calls' plans, one after the other (owned)
    // The no-allocation entry point: this device's scratch array (its device
    // address, from hipGetSymbolAddress at creation) and, during such a
    // call, the arena carved from it.
    void *scratchPtr = nullptr;
    // Host memory the packed score kernel raises when a strip's wait runs
    // past its bound (never expected).
    uint32_t *waitFlag = nullptr;
    Arena arena;
    bool noAlloc = false;   // inside sqmi_align_score_noalloc
    // The last sqmi_align_score call, kept for an identical next call: the
    // key of its inputs, its statistics and its launches; more than
    // kDirectLaunches of them, from the second such call on, as an instantiated
    // HIP graph (to capture and instantiate one takes 60-80 us, which a call that
    // comes once does not get back).  Its plan lives on in the context's device
    // buffers, so any other call on the context drops it.
    struct Replay {
        bool valid = false;
        uint64_t key = 0;
        std::vector<std::function<hipError_t()>> launches;   // until a graph holds them
        hipGraphExec_t exec = nullptr;
        sqmi_stats stats{};
    } replay;
};

namespace {

sqmi_status fail(sqmi_context *ctx, sqmi_status st, const std::string &msg)
{
    if (ctx)
        ctx->lastError = msg;
    return st;
}

sqmi_status hipFail(sqmi_context *ctx, hipError_t err, const char *what)
{
    // The runtime keeps an error until it is read: without this the next
    // call's check after a launch would report it again.
    (void)hipGetLastError();
    std::string msg = std::string(what) + ": " + hipGetErrorString(err);
    return fail(ctx, err == hipErrorOutOfMemory ? SQMI_ERR_OUT_OF_MEMORY : SQMI_ERR_DEVICE, msg);
}

void endView(DevBuf &b)
{
    if (!b.view)
        return;
    b.p = b.own;
    b.cap = b.ownCap;
    b.view = false;
}

hipError_t ensure(DevBuf &b, size_t bytes)
{
    if (bytes == 0)
        bytes = 16;
    endView(b);
    if (b.cap >= bytes)
        return hipSuccess;
    if (b.arena) {
        // 256-byte aligned pieces of the arena; an outgrown piece stays unused.
        const size_t need = (bytes + 255) & ~(size_t)255;
        if (b.arena->used + need > b.arena->cap)
            return hipErrorOutOfMemory;
        b.p = b.arena->base + b.arena->used;
        b.arena->used += need;
        b.cap = need;
        return hipSuccess;
    }
    if (b.p)
        (void)hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
    hipError_t e = hipMalloc(&b.p, bytes);
    if (e == hipSuccess)
        b.cap = bytes;
    return e;
}

// Launches collected during a call's preparation and run (or captured into
// a HIP graph) once every upload is enqueued.
using Deferred = std::vector<std::function<hipError_t()>>;

// SQMI_GRAPH=0 turns off the replay of identical sqmi_align_score calls.
bool graphsEnabled()
{
    const char *env = std::getenv("SQMI_GRAPH");
    return !(env && *env == '0');
}

void dropReplay(sqmi_context *ctx)
{
    if (ctx->replay.exec)
        (void)hipGraphExecDestroy(ctx->replay.exec);
    ctx->replay = sqmi_context::Replay{};
}

// A replayed call of up to this many launches runs them one by one: a graph of
// two takes 8-10 us longer than they do.
constexpr size_t kDirectLaunches = 4;

// The kept launches as an instantiated graph; a capture the runtime refuses
// leaves them to be run one by one.
void captureReplay(sqmi_context *ctx)
{
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    if (hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal) == hipSuccess) {
        hipError_t err = hipSuccess;
        for (auto &f : ctx->replay.launches)
            if (err == hipSuccess)
                err = f();
        const hipError_t end = hipStreamEndCapture(ctx->stream, &graph);
        if (err == hipSuccess && end == hipSuccess && graph && hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) == hipSuccess)
            ctx->replay.exec = exec;
        if (graph)
            (void)hipGraphDestroy(graph);
    }
    (void)hipGetLastError();   // a refused capture leaves its error behind
}

uint64_t mix64(uint64_t x)
{
    x ^= x >> 33;
    x *= 0xff51afd7ed558ccdULL;
    x ^= x >> 33;
    x *= 0xc4ceb9fe1a85ec53ULL;
    x ^= x >> 33;
    return x;
}

// Order-sensitive 64-bit digest of n int64 values (a sum of position-tagged
// mixes, so threads can take contiguous ranges).
uint64_t digest64(const int64_t *a, int64_t n)
{
    uint64_t h = 0;
#pragma omp parallel for schedule(static) reduction(+ : h) if (n > 65536)
    for (int64_t i = 0; i < n; ++i)
        h += mix64((uint64_t)a[i] ^ ((uint64_t)i * 0x9e3779b97f4a7c15ULL));
    return mix64(h ^ (uint64_t)n);
}

// Bytes an arena piece of `bytes` takes (ensure() rounds to 256).
size_t arenaBytes(size_t bytes) { return ((bytes ? bytes : 16) + 255) & ~(size_t)255; }

void release(DevBuf &b)
{
    endView(b);
    if (b.p && !b.arena)
        (void)hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
}

// Staged uploads.  A call's small arrays (offsets, tables, work lists) are
// gathered in pinned memory and sent together: a copy from pageable memory
// takes 8-12 us each, whatever its size, and large ones run at one thread's
// memcpy.  Results come back the same way (20 MB to pageable memory 1.13 ms,
// to pinned memory 0.38 and 0.03 from there).  stageBegin: `bytes` bounds what
// the call will put (each array rounded up to 256 bytes), `down` what it will
// fetch.  The pinned memory stays with the context, so it has a bound: results
// past kMaxDown go straight to the caller's memory, of uploads past kMaxUp
// (about 10 million pairs) the arrays that do not fit are copied by themselves;
// without pinned or device memory for the stage all are.  SQMI_STAGE_MB sets
// both bounds (0: no staging; tests).
constexpr size_t kMaxUp = (size_t)512 << 20, kMaxDown = (size_t)256 << 20;

// stageResume: a call that replays the last one's launches; what that one put
// stays in place, results have `down` bytes of the pinned memory that is there.
hipError_t stageResume(sqmi_context *ctx, size_t down)
{
    ctx->pinOn = false;
    ctx->downUsed = 0;
    ctx->downCap = down <= std::min(ctx->pinCap, kMaxDown) ? down : 0;
    ctx->down.clear();
    if (ctx->pinBusy) {   // an earlier call failed between its uploads and its end
        const hipError_t e = hipDeviceSynchronize();
        if (e != hipSuccess)
            return e;
        ctx->pinBusy = false;
    }
    return hipSuccess;
}

hipError_t stageBegin(sqmi_context *ctx, size_t bytes, size_t down = 0)
{
    const hipError_t e = stageResume(ctx, 0);
    if (e != hipSuccess)
        return e;
    size_t maxUp = kMaxUp, maxDown = kMaxDown;
    if (const char *env = std::getenv("SQMI_STAGE_MB"))
        if (*env)
            maxUp = maxDown = (size_t)std::max(0ll, std::min(512ll, std::atoll(env))) << 20;
    if (ctx->noAlloc || maxUp == 0)
        return hipSuccess;
    bytes = std::min(bytes, maxUp);
    if (down > maxDown)
        down = 0;
    const size_t most = std::max(bytes, down);
    if (ctx->pinCap < most) {
        if (ctx->pin)
            (void)hipHostFree(ctx->pin);
        ctx->pin = nullptr;
        ctx->pinCap = 0;
        const size_t cap = std::min(most + most / 4, kMaxUp);
        void *p = nullptr;
        if (hipHostMalloc(&p, cap, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            return hipSuccess;
        }
        ctx->pin = static_cast<char *>(p);
        ctx->pinCap = cap;
    }
    if (ensure(ctx->stage, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return hipSuccess;
    }
    ctx->downCap = down;
    ctx->pinUsed = ctx->pinSent = 0;
    ctx->pinOn = true;
    return hipSuccess;
}

// Whether the stage has room for `bytes` more.
bool stageFits(const sqmi_context *ctx, size_t bytes)
{
    return ctx->pinOn && ctx->pinUsed + bytes <= std::min(ctx->pinCap, ctx->stage.cap);
}

// Sends what has been put since the last flush.
hipError_t stageFlush(sqmi_context *ctx)
{
    if (!ctx->pinOn || ctx->pinSent == ctx->pinUsed)
        return hipSuccess;
    ctx->pinBusy = true;
    const hipError_t e = hipMemcpyAsync(static_cast<char *>(ctx->stage.p) + ctx->pinSent, ctx->pin + ctx->pinSent,
                                        ctx->pinUsed - ctx->pinSent, hipMemcpyHostToDevice, ctx->stream);
    ctx->pinSent = ctx->pinUsed;
    return e;
}

// The call's stream is synchronised.
void stageEnd(sqmi_context *ctx) { ctx->pinOn = ctx->pinBusy = false; }

size_t stageBytes(size_t bytes) { return (bytes + 255) & ~(size_t)255; }

// A host copy, by all threads from 2 MB on.
constexpr size_t kParallelCopy = (size_t)2 << 20;
void copyBytes(void *dst, const void *src, size_t len)
{
    if (len < kParallelCopy) {
        if (len)
            std::memcpy(dst, src, len);
        return;
    }
    constexpr size_t kPart = (size_t)512 << 10;
    const int64_t parts = (int64_t)((len + kPart - 1) / kPart);
#pragma omp parallel for schedule(static)
    for (int64_t q = 0; q < parts; ++q)
        std::memcpy(static_cast<char *>(dst) + q * kPart, static_cast<const char *>(src) + q * kPart,
                    std::min(kPart, len - (size_t)q * kPart));
}

// dst receives src[0 .. bytes) of device memory by the next deliver() after a
// synchronisation of the stream.  (The uploads from the same pinned memory
// precede the results in the stream.)
hipError_t fetch(sqmi_context *ctx, void *dst, const void *src, size_t bytes)
{
    if (ctx->downUsed + stageBytes(bytes) > ctx->downCap)
        return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream);
    ctx->down.push_back({dst, ctx->pin + ctx->downUsed, bytes});
    ctx->pinBusy = true;
    const hipError_t e = hipMemcpyAsync(ctx->pin + ctx->downUsed, src, bytes, hipMemcpyDeviceToHost, ctx->stream);
    ctx->downUsed += stageBytes(bytes);
    return e;
}

// The first n fetched arrays, to their places.
void deliver(sqmi_context *ctx, size_t n)
{
    for (size_t k = 0; k < n; ++k)
        copyBytes(ctx->down[k].dst, ctx->down[k].src, ctx->down[k].bytes);
    ctx->down.erase(ctx->down.begin(), ctx->down.begin() + n);
}
void deliver(sqmi_context *ctx) { deliver(ctx, ctx->down.size()); }

struct Piece {
    const void *src;
    size_t bytes;
};

// b holds the pieces, one after the other, in device memory once the stage is
// flushed (or, where the call does not stage or they do not fit, once the
// stream has run the copies).
hipError_t put(sqmi_context *ctx, DevBuf &b, const Piece *pieces, size_t n)
{
    size_t bytes = 0, at = 0;
    for (size_t k = 0; k < n; ++k)
        bytes += pieces[k].bytes;
    if (!stageFits(ctx, stageBytes(bytes))) {
        hipError_t e = ensure(b, bytes);
        for (size_t k = 0; k < n && e == hipSuccess; at += pieces[k++].bytes)
            if (pieces[k].bytes)
                e = hipMemcpyAsync(static_cast<char *>(b.p) + at, pieces[k].src, pieces[k].bytes, hipMemcpyHostToDevice,
                                   ctx->stream);
        return e;
    }
    endView(b);
    b.own = b.p;
    b.ownCap = b.cap;
    b.view = true;
    b.p = static_cast<char *>(ctx->stage.p) + ctx->pinUsed;
    b.cap = bytes;
    char *dst = ctx->pin + ctx->pinUsed;
    ctx->pinUsed += stageBytes(bytes);
    for (size_t k = 0; k < n; at += pieces[k++].bytes)
        copyBytes(dst + at, pieces[k].src, pieces[k].bytes);
    // Large arrays are on their way while the next one is gathered.
    return bytes < kParallelCopy ? hipSuccess : stageFlush(ctx);
}
hipError_t put(sqmi_context *ctx, DevBuf &b, const void *src, size_t bytes)
{
    const Piece one{src, bytes};
    return put(ctx, b, &one, 1);
}

// New contents for two buffers that the last call put, in one copy.
hipError_t restage(sqmi_context *ctx, const DevBuf &a, const void *srcA, size_t bytesA, const DevBuf &b, const void *srcB,
                   size_t bytesB)
{
    char *stage = static_cast<char *>(ctx->stage.p);
    const size_t atA = static_cast<char *>(a.p) - stage, atB = static_cast<char *>(b.p) - stage;
    copyBytes(ctx->pin + atA, srcA, bytesA);
    copyBytes(ctx->pin + atB, srcB, bytesB);
    const size_t from = std::min(atA, atB), to = std::max(atA + bytesA, atB + bytesB);
    ctx->pinBusy = true;
    return hipMemcpyAsync(stage + from, ctx->pin + from, to - from, hipMemcpyHostToDevice, ctx->stream);
}

struct ScoringInfo
{
    int alpha = 0;
    int o = 0, e = 0;
    int sMax = 0, sMin = 0;
    bool dna = false;   // v_perm profile path possible
    bool dnaDrift = false;   // and for the drifted scores t + drift (global score kernels)
};

// The score kernels' drifted representation (kernels.hpp, Drift; local:
// score16.hpp).  Scores t below 0 raise the bias, so that a diagonal step
// never leaves the value range.
Drift driftOf(const ScoringInfo &si, bool local)
{
    Drift r;
    const int ext = std::max(si.o, si.e);
    r.d = -ext;
    r.cost = ext - si.o;
    const int tMin = std::min(0, si.sMin - si.o - (local ? 0 : ext));
    if (local) {
        r.bias = r.cost + 2 * r.d + 2 - tMin;
        r.neg = r.bias - r.cost;
    } else {
        r.neg = r.cost - tMin + 1;
        r.bias = r.neg + 3 * r.cost + 1;
    }
    return r;
}

// Whether a pair's stored values stay within kDriftNarrowMax (and no t is
// below 0): at most bias + sMax * min(n, m) + drift * (n + m), local + drift
// * 17 instead.  Pairs inside the int16 window (fitsInt16) always stay within
// 65535: there sMax * min(n, m) is at most 30719 and drift * (n + m) at most
// 26624, the bias of costs up to 1024 at most 6146 (local: 17 * 1024 and 4098).
bool driftNarrow(const ScoringInfo &si, const Drift &dr, bool local, int64_t n, int64_t m)
{
    const int64_t span = local ? 17 : n + m + 2 * kDriftSlack;
    return dr.neg == (local ? 2 * dr.d + 2 : dr.cost + 1) &&
           dr.bias + (int64_t)std::max(0, si.sMax) * (std::min(n, m) + kDriftSlack) + dr.d * span <= kDriftNarrowMax;
}

// What a path inside a band of W1 + 1 diagonals can lose, in drifted values,
// on the way to a cell up to maxM rows down: no more than by gaps of the
// band's width right and down in turn, or by mismatches along a diagonal.
// (The plain bias covers two gaps, which reach any cell of a whole matrix.)
int64_t bandDrop(const ScoringInfo &si, const Drift &dr, int64_t W1, int64_t maxM)
{
    const int64_t zigzag = dr.cost * (2 * ((maxM + W1 - 1) / W1) + 6);
    const int64_t diagonal = std::max<int64_t>(0, -((int64_t)si.sMin + 2 * dr.d)) * maxM + 3 * dr.cost;
    return std::min(zigzag, diagonal);
}

// Conservative range of every value a pair can produce inside the DP (H, E, F
// and H + gapOpen), from the sizes alone.  H <= max(0, sMax) * min(n, m) since
// gap costs are <= 0.  H(i,j) >= the score of the all-gap path along row 0
// and column j, 2*o + (i+j-2)*max(o,e) (a gap chain grows by max(o,e) per
// character); E, F and H + o are at least H + o; the diagonal term at least
// H + sMin.
bool fitsInt16(const ScoringInfo &si, int64_t n, int64_t m, bool local)
{
    const int64_t up = (int64_t)std::max(0, si.sMax) * std::min(n, m);
    const int64_t lowH = local ? 0 : 2LL * si.o + (n + m) * (int64_t)std::min(std::max(si.o, si.e), 0);
    const int64_t low = lowH + std::min({si.o, si.sMin, 0}) + std::min(si.e, 0);
    return up <= 32767 - kGuard16 && low >= (int64_t)kNeg16 + kGuard16 && n <= 30000 && m <= 30000;
}

// The same bound for the tiled int32 kernels of long pairs, whose minus
// infinity is -2^29: every real value stays within +-2^28.
bool fitsLong32(const ScoringInfo &si, int64_t n, int64_t m)
{
    const int64_t up = (int64_t)std::max(0, si.sMax) * std::min(n, m);
    const int64_t lowH = 2LL * si.o + (n + m) * (int64_t)std::min(std::max(si.o, si.e), 0);
    const int64_t low = lowH + std::min({si.o, si.sMin, 0}) + std::min(si.e, 0);
    return up < (1LL << 28) && low > -(1LL << 28) && n < (1LL << 30) && m < (1LL << 30);
}

// The pairs of one shape: for groups of 16 or 64 lanes the items become units
// of the packed score kernel (Planned::units), for the one-pair-per-lane and
// trace kernels they are launched as they are.
struct Plan16
{
    Variant16 var;
    std::vector<int32_t> order;
    std::vector<WorkItem> items;
    int maxN = 0;
};

int pairsPerWave(const Variant16 &v) { return 2 * (64 / v.G); }

// Shapes of the score calls: a pair couple per 16 or 64 lanes (kScore16) or
// per lane (kLane16).
bool shapeSupported(const Variant16 &v)
{
    if (v.G == 1)
        return laneSupported(v);
    return (v.G == 16 && (v.R == 8 || v.R == 16)) || (v.G == 64 && (v.R == 4 || v.R == 8 || v.R == 16));
}

// The planner's table (seqan_amd/tuning/shapes.json, turned into C++ by the
// build): per category (DNA byte profile or substitution table, global or
// local), length bin b (2^(b-1) < |V| + 1 <= 2^b) and count class (the call's
// pairs on the packed route, at least kTabCountClasses[c]), an index into
// kTabShapes: groups (0, 0) or one pair couple per lane (1, rows).
#include "shape_table.inc"

int lengthBin(int64_t m)
{
    // The smallest b <= 15 with 2^b >= m + 1.
    if (m < 1)
        return 0;
    const int b = 64 - __builtin_clzll((unsigned long long)m);
    return b < 15 ? b : 15;
}

int shapeCategory(bool dna, bool local) { return (dna ? 0 : 2) + (local ? 1 : 0); }

// SQMI_SHAPE_RULE=fixed: groups of 16 lanes and whole items for every pair,
// for comparing the shape rules with one shape.
bool fixedShapeRule()
{
    const char *env = std::getenv("SQMI_SHAPE_RULE");
    return env && std::strcmp(env, "fixed") == 0;
}

// Whether the shape table gives length bin `bin` the one-pair-per-lane
// kernel, for a call holding pairs16 pairs on the packed route (all bins: the
// launches run side by side, so the whole call is what fills the GPU), and
// its rows per lane.
int laneRows(int category, int bin, int64_t pairs16)
{
    int cls = 0;
    while (cls + 1 < kTabNClasses && pairs16 >= kTabCountClasses[cls + 1])
        ++cls;
    const int idx = kTabChoice[category][bin][cls];
    return kTabShapes[idx][0] == 1 ? kTabShapes[idx][1] : 0;
}

// Lanes per pair couple and whole items or strips, by the time a pair takes
// against the whole call's.  A wave of 16-lane groups sweeps n x m cells (of
// eight pairs at once) in about 5.7 n m cycles at three waves per SIMD, a wave
// of one 64-lane group (one couple) in a quarter of that; the call's cells
// take about 2.3e-4 cycles each on the whole chip.  An item may take a
// quarter of the call's time: longer ones end after the others have left the
// chip.  So couples go to 64 lanes from 1.0e-5 of the call's cells on, and
// their row blocks to different waves (strips) from 4e-5 on.  Measured (MI355X):
// 3,001 uneven pairs (100 bp - 10 kbp, semi-global) 14.2 -> 1.8 ms, where four
// waves of one workgroup used to share an item's blocks; 1,048,576 of them
// 99 -> 69 ms, of which the shorter recurrence gives most.
constexpr double kCouple64Share = 1.0e-5, kStripShare = 4.0e-5;
// Device memory of a score call's strips, at most (and SQMI_TRACE_BUDGET_MB):
// the shares alone let 25,000 pairs of 13 kbp take 17 GB.  (16,000 of 13 kbp,
// all strips, 11 GB: 330 ms; within 4 GB: 291.)
constexpr int64_t kMaxStripBytes = (int64_t)4 << 30;
// Time of a strip's step (ns), by its rows per lane: alone on a SIMD, and of a full one.
struct LongCost {
    int rows;
    double alone, full;
};
constexpr LongCost kLongCosts[] = {{4, 115, 63}, {8, 153, 111}, {16, 230, 203}};
// Waves of a workgroup of the packed banded kernel, by its ring's columns: the
// ring is the band and a block, and a wave follows the one above by R + 8
// columns.  (Rings past 256 columns: four waves with rings of their own.)
int bandWaves(int cols) { return cols > 256 ? 4 : cols > 128 ? 8 : cols > 64 ? 4 : 2; }
// Banded scores, ns: a column of a packed item's block, by one wave (rings in
// memory) and with 2, 4 and 8 waves sharing the item; a row of a pair on the
// int32 kernels, alone and per SIMD of a full chip (wide: of 64 diagonals).
// 1,000 / 4,096 / 16,384 / 65,536 pairs, free ends, 1 kbp, 201 diagonals: packed
// 0.81 / 0.81 / 0.84 / 2.5 ms, int32 2.5 / 3.3 / 12.8 / 51.5; local, 150 bp,
// 33 diagonals: 0.11 / 0.11 / 0.11 / 0.18 against 0.04 / 0.06 / 0.19 / 0.68.
constexpr double kBandColumnAlone = 335, kBandColumn[3] = {170, 80, 60}, kBandNarrowLone = 270, kBandNarrowFull = 70, kBandWideLone = 615, kBandWideFull = 202;
// Waves of the packed score kernel that the chip holds (256 CUs, 4 SIMDs, 3).
constexpr int64_t kResidentWaves = 3072;
// Calls of pairs of about one size (the largest at most four times the mean):
// 64 lanes for all of them cost more than twice the instructions, their skew
// of 64 steps weighs on short pairs, and four times the units and more (strips)
// are claimed one by one.  In cycles: a pair alone on 16 lanes about 3.2 a cell,
// with the table 4 (more waves per SIMD: up to twice that), on 64 lanes 0.93
// (1.2), the skew and 4,000; 40 a unit.  Whether 16 lanes are the faster.  Device us, 64
// lanes / 16: 4,096 pairs of 20-60 bp 66 / 31, of 66-126 71 / 43, of 150 76 / 61, of
// 100-200 80 / 77, of 400 205 / 203; 2,048 of 66-126 46 / 40, of 150 53 / 55, of 200
// 60 / 77; 53,121 of 68 bp, local, 413 / 152; 20,000 of 300 bp 413 / 348.  Proteins:
// 4,096 of 66-126 78 / 54, of 100-200 84 / 107, of 300 198 / 189; 8,192 of 200-400
// 236 / 345; 62,172 of 50-372 by 50-744, local, 1,350 / 1,020.  Past 512 rows (mean)
// 64 lanes have rows enough to cost the same: 20,000 of 1 kbp, global, 2,240 / 2,420.
bool evenOn16(double most, double pairs, double cells, bool dna)
{
    const double alone16 = dna ? 3.2 : 4.0, alone64 = dna ? 0.93 : 1.2, side = std::max(1.0, std::sqrt(most));
    const double waves = pairs / 8 / 1024, skew = (side + 64) / side;
    double blocks = pairs * kStripShare < 1 ? std::ceil((side + 1) / 256) : 1;   // makeUnits: strips of 4 rows per lane, or more
    while (blocks > 1 && blocks * pairs / 2 > 2 * kResidentWaves)
        blocks = std::ceil(blocks / 2);
    const double t16 = std::max(alone16 * most * std::max(1.0, 0.66 * std::min(3.0, waves)), 2.3e-4 * cells) + 40 * pairs / 8;
    const double t64 = std::max(alone64 * most, 2.1 * 2.3e-4 * cells) * skew + 40 * blocks * pairs / 2 + 4000;
    return cells <= 512.0 * 512.0 * pairs && 1.03 * t64 >= t16;
}
// Global pairs whose drifted values need all 16 bits (Variant16::wide), one per
// lane with 32 rows: in the length bins up to kWideLane[k].bin when the call
// holds that many of them there, `alone` or beside pairs that stay on groups
// (the lane kernel's sweep of its longest pair then comes on top).  Device ms,
// match 1, mismatch -4, gaps -1 / -2, global and all ends free, groups -> lanes: 524,288 pairs
// of 30-40 bp 0.92 / 0.98 -> 0.31 / 0.37; 20,000 of 10-20 bp 0.08 / 0.08 -> 0.05 / 0.07;
// 30,000 of 17-30 bp 0.09 / 0.09 -> 0.06 / 0.09; of 34-62 bp 131,072 0.28 / 0.28 ->
// 0.18 / 0.24 and 60,000 0.16 / 0.17 -> 0.17 / 0.22; of 66-126 bp 262,144 0.80 / 0.83 ->
// 0.72 / 0.76 and 131,072 0.43 / 0.47 -> 0.56 / 0.66.
struct WideLane {
    int bin;
    int64_t alone, beside;
};
constexpr WideLane kWideLane[] = {{7, 262144, 1048576}, {6, 131072, 262144}, {5, 24576, 65536}, {4, 16384, 49152}};
// Rows per unit of the group shapes' row counts.
constexpr int kUnitRows = 64;
inline int64_t unitsOfRows(int64_t m) { return (m + kUnitRows) / kUnitRows; }   // m + 1 rows

// Row blocks of a pair with m rows under shape v (at most 255 fit the keys).
// Row blocks of G * R rows (a power of two for every compiled shape).
int64_t blocksFor(const Variant16 &v, int64_t m)
{
    const int64_t br = (int64_t)v.G * v.R;
    return (br & (br - 1)) == 0 ? (m + br) >> __builtin_ctzll((unsigned long long)br) : (m + br) / br;
}

// Calls with at most this many pairs plan on one thread: waking the thread
// team costs more than it saves.
constexpr int64_t kParallelMin = 32768;

sqmi_status checkSet(sqmi_context *ctx, const sqmi_sequences *s, const char *name)
{
    if (!s)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, std::string(name) + " is null");
    if (s->count < 0)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, std::string(name) + ": negative count");
    if (s->count > 0 && (!s->offsets || !s->residues))
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, std::string(name) + ": null offsets or residues");
    if (s->count > INT32_MAX - 1)
        return fail(ctx, SQMI_ERR_UNSUPPORTED, std::string(name) + ": more than 2^31-2 sequences");
    if (s->count > 0 && s->offsets[0] < 0)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, std::string(name) + ": negative offset");
    const int64_t n = s->count;
    const int64_t *off = s->offsets;
    bool bad = false;
#pragma omp parallel for schedule(static) reduction(|| : bad) if (n > kParallelMin)
    for (int64_t i = 0; i < n; ++i)
        bad = bad || off[i + 1] < off[i];
    if (bad)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, std::string(name) + ": offsets not monotone");
    return SQMI_OK;
}

double msSince(std::chrono::steady_clock::time_point t0)
{
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

struct Key
{
    uint32_t key;
    int32_t id;
};

// A vector whose new elements are left uninitialised: the planner's large
// arrays are written in full, in parallel, right after they are sized.
template <class T>
struct RawAlloc : std::allocator<T>
{
    template <class U>
    struct rebind { using other = RawAlloc<U>; };
    template <class U>
    void construct(U *p) noexcept { ::new (static_cast<void *>(p)) U; }
    template <class U, class... A>
    void construct(U *p, A &&...a) { ::new (static_cast<void *>(p)) U(std::forward<A>(a)...); }
};
template <class T>
using RawVec = std::vector<T, RawAlloc<T>>;

struct Planned
{
    ScoringInfo si;
    uint32_t flags = 0;
    bool local = false;
    uint32_t mode = 0;
    uint32_t track = 0;
    std::vector<int32_t> emptyIds, ids32;
    std::vector<int32_t> idsLong;   // int32 pairs for the tiled long-pair kernels
    std::vector<int64_t> scratchOff32;
    int64_t scratch32 = 0;
    RawVec<Key> keys16, keysTmp;    // int16 pairs, sorted by bucket key; the sort's other half
    std::vector<uint32_t> sortHist;
    std::vector<Variant16> shapes;  // int16 shape slots (key classes 0..)
    std::vector<Plan16> plans;      // one per one-pair-per-lane or trace shape in use
    // Packed score kernel: pair ids grouped by item, units, buffers.
    RawVec<int32_t> order16;
    RawVec<ScoreUnit> units;
    int64_t slotWords = 0, stripWords = 0;
    int64_t items16 = 0, padded16 = 0;
    bool dna16 = false;             // profile path of the packed kernels
    Drift drift{};
    int64_t cells = 0;

    // Back to an empty plan that keeps its arrays (a context's calls share
    // one, so that large calls don't fault their pages in every time).
    void reset()
    {
        emptyIds.clear();
        ids32.clear();
        idsLong.clear();
        scratchOff32.clear();
        shapes.clear();
        plans.clear();
        scratch32 = slotWords = stripWords = items16 = padded16 = cells = 0;
    }

    // Back to an empty plan of its own after a call whose arrays a context
    // should not keep: past 128 MB (some 5 million pairs) faulting them in
    // again is a small part of the next such call.
    static constexpr size_t kKeepBytes = (size_t)128 << 20;
    void trim()
    {
        auto of = [](const auto &v) { return v.capacity() * sizeof(v[0]); };
        size_t bytes = of(emptyIds) + of(ids32) + of(idsLong) + of(scratchOff32) + of(keys16) + of(keysTmp) + of(order16) + of(units);
        for (const Plan16 &p : plans)
            bytes += of(p.order) + of(p.items);
        if (bytes > kKeepBytes)
            *this = Planned{};
    }
};

// Trims the context's plan when the call ends.
struct PlanUse {
    Planned &p;
    ~PlanUse() { p.trim(); }
};

// The packed long-pair kernels (long16.hip) hold values relative to a base;
// target: where a strip's top row is kept; a strip of 64 R rows needs every
// value below kDriftNarrowMax, the cells of a wave growing by at most sMax + 2
// drift per row and column.
int longTarget(const ScoringInfo &si, const Drift &dr)
{
    return dr.neg + 8 * dr.cost + 64 * (std::max(si.sMax, 0) + 2 * dr.d) + 16;
}
bool longRowsFit(const ScoringInfo &si, int R)
{
    const Drift dr = driftOf(si, false);
    const int64_t grow = std::max(si.sMax, 0) + 2 * (int64_t)dr.d;
    return si.dnaDrift && si.o <= 0 && si.e <= 0 && dr.neg == dr.cost + 1 &&
           longTarget(si, dr) + kLongSlackV + (64 * R + 256 + kLongT) * grow + 8 * dr.cost <= kDriftNarrowMax;
}
bool longPacked(const ScoringInfo &si, uint32_t flags) { return !(flags & SQMI_FORCE_INT32) && longRowsFit(si, 4); }

// Test and tuning switch: SQMI_LONG_ALL=1 sends every pair the long route
// can take there, also those the packed kernels could score.
bool longAll()
{
    const char *env = std::getenv("SQMI_LONG_ALL");
    return env && *env == '1';
}

bool envFlag(const char *name)
{
    const char *env = std::getenv(name);
    return env && *env == '1';
}

// Pairs outside the int16 window whose sides are both at least this long (and
// that are DNA) run the long-pair kernels instead of one thread per pair (2048,
// or SQMI_LONG_MIN_SIDE).
int64_t longMinSide()
{
    const char *env = std::getenv("SQMI_LONG_MIN_SIDE");
    if (env && *env && std::atoll(env) > 0)
        return std::atoll(env);
    return 2048;
}

// After a call's final synchronisation: whether a strip's wait ran past its
// bound (the flag is raised by the kernel, in host memory).
sqmi_status stripCheck(sqmi_context *ctx)
{
    if (*static_cast<volatile uint32_t *>(ctx->waitFlag) == 0)
        return SQMI_OK;
    *ctx->waitFlag = 0;
    return fail(ctx, SQMI_ERR_DEVICE, "a row block's wait for the one above it ran past its bound; results are not valid");
}

// Streams the long-pair forward spreads its pair couples over (1..4).  On
// 64 pairs of 100 kbp with 128-column tiles: 1 stream 263 ms, 2 streams
// 164 ms, 3 streams 157 ms (with 256-column tiles: 220, 170, 170 ms; 4
// streams 260 ms, the 4th sharing a hardware queue); starting the groups
// some anti-diagonals apart only made it slower.
int longStreams()
{
    const char *env = std::getenv("SQMI_LONG_STREAMS");
    const int v = (env && *env) ? std::atoi(env) : 3;
    return std::max(1, std::min(v, sqmi_context::kMaxLongStreams));
}


// Stable LSD radix sort of 28-bit keys in two passes of 14 bits, each pass
// split into contiguous per-thread ranges so that equal digits keep their
// input order.
void radixSort(RawVec<Key> &keys, RawVec<Key> &tmp, std::vector<uint32_t> &hist)
{
    const size_t n = keys.size();
    if (n < 2)
        return;
    if (n <= 1024) {   // clearing and summing the digit counts takes longer (30 us)
        std::stable_sort(keys.begin(), keys.end(), [](const Key &a, const Key &b) { return a.key < b.key; });
        return;
    }
    tmp.resize(n);
    int T = 1;
#ifdef _OPENMP
    T = std::max(1, std::min(omp_get_max_threads(), (int)(n / 16384) + 1));
#endif
    constexpr int B = 14, NB = 1 << B;
    hist.resize((size_t)T * NB);
    for (int shift = 0; shift < 2 * B; shift += B) {
        const uint32_t mask = (uint32_t)NB - 1;
#pragma omp parallel num_threads(T)
        {
            int t = 0;
#ifdef _OPENMP
            t = omp_get_thread_num();
#endif
            const size_t lo = n * t / T, hi = n * (t + 1) / T;
            uint32_t *h = hist.data() + (size_t)t * NB;
            std::fill(h, h + NB, 0u);
            for (size_t k = lo; k < hi; ++k)
                ++h[(keys[k].key >> shift) & mask];
#pragma omp barrier
#pragma omp single
            {
                // One thread: the sums of one array.  (The nested loop took 7 to
                // 20 us more for its 2 x 16,384 digits, by where the compiler
                // put its branches: 4,096 pairs of 150 bp 169 us, so 154.)
                uint32_t run = 0;
                if (T == 1) {
                    for (int d = 0; d < NB; ++d) {
                        const uint32_t v = h[d];
                        h[d] = run;
                        run += v;
                    }
                } else {
                    for (int d = 0; d < NB; ++d)
                        for (int u = 0; u < T; ++u) {
                            uint32_t &c = hist[(size_t)u * NB + d];
                            const uint32_t v = c;
                            c = run;
                            run += v;
                        }
                }
            }
            for (size_t k = lo; k < hi; ++k)
                tmp[h[(keys[k].key >> shift) & mask]++] = keys[k];
        }
        keys.swap(tmp);
    }
}

// Bucket keys (28 bits): class (3 bits: 0..6 int16 shape slot, 7 int32 or
// empty) | 1023 - row units (10 bits) | 32767 - |H| (15 bits).  Ascending
// order puts int16 pairs first, grouped by shape and row units (most first),
// widest first, then the int32 and empty pairs in input order.  A row
// unit is 64 rows for the group shapes (their block 0 is as tall as the item
// needs), a whole block for the one-pair-per-lane and the trace kernels.
constexpr int kKeyNBits = 15, kKeyUnitBits = 10, kKeyClassShift = kKeyNBits + kKeyUnitBits;
constexpr uint32_t kClassRest = 7;
// Shape slots of the score calls: group shapes (the longest pairs first; + 0
// wide values, + 1 narrow), then lanes.
constexpr uint32_t kSlot64 = 0, kSlot16 = 2, kSlotLane16 = 4, kSlotLane32 = 5, kSlotLaneWide = 6;
constexpr int64_t kMaxBlocks16 = 255;   // row blocks per pair of a packed work item
inline uint32_t bucketOf(uint32_t key) { return key >> kKeyNBits; }
inline int32_t widthOf(uint32_t key) { return (int32_t)((1u << kKeyNBits) - 1 - (key & ((1u << kKeyNBits) - 1))); }
inline int32_t unitsOf(uint32_t key) { return (int32_t)(1023u - ((key >> kKeyNBits) & 1023u)); }
// Row units of the group shapes: 64 rows (fine), or 256 (coarse: units rounded
// up to 4).  Fine units cut the rows of block 0 but split the pairs of a
// length bin over 4 times as many buckets, which widens the spread of |H|
// inside an item when the bin holds few pairs; so a bin takes fine units from
// kFineUnitPairs pairs on (SQMI_ROW_UNITS=block / quarter: always coarse /
// fine).
constexpr int64_t kFineUnitPairs = 8192;
int rowUnitsMode()   // 0 by bin size, 1 coarse, 2 fine
{
    const char *env = std::getenv("SQMI_ROW_UNITS");
    if (env && std::strcmp(env, "block") == 0)
        return 1;
    if (env && std::strcmp(env, "quarter") == 0)
        return 2;
    return 0;
}
// Work items with at least this many row blocks become strips
// (SQMI_COOP_MIN_BLOCKS; 0: none, unset: the rule of kStripShare).
int stripMinBlocks()
{
    const char *env = std::getenv("SQMI_COOP_MIN_BLOCKS");
    return env && *env ? std::max(0, std::atoi(env)) : -1;
}

// Strips in the order a wave should claim them: by the steps from a strip's
// start to its item's end (its columns, and kStripLag for every block from it
// on), the most first.  The strip above always comes earlier.  Claimed item
// by item, an item's lower strips held waves that only waited for the upper
// ones.  The whole items follow in their order.  Rows of 8,192 protein
// pairs, local: trace kernel 3.35 -> 2.9 ms.  (Score calls measured the same
// either way and keep their items' order.)
constexpr int32_t kStripLag = 128;
void orderStrips(RawVec<ScoreUnit> &units, size_t begin)
{
    constexpr int kShift = 3, kBuckets = 1 << 13;   // 8 steps per bucket, up to 65,536 steps
    auto bucket = [](const ScoreUnit &u) {
        const int64_t left = u.maxN + (int64_t)kStripLag * (u.nblocks - u.block);
        return u.block < 0 ? kBuckets : kBuckets - 1 - (int)std::min<int64_t>(left >> kShift, kBuckets - 1);
    };
    bool strips = false;
    for (size_t k = begin; k < units.size() && !strips; ++k)
        strips = units[k].block > 0;
    if (!strips)
        return;
    std::vector<uint32_t> at(kBuckets + 2, 0);
    for (size_t k = begin; k < units.size(); ++k)
        ++at[bucket(units[k]) + 1];
    for (int b = 0; b <= kBuckets; ++b)
        at[b + 1] += at[b];
    const std::vector<ScoreUnit> from(units.begin() + begin, units.end());
    for (const ScoreUnit &u : from)
        units[begin + at[bucket(u)]++] = u;
}

// Units of the packed score kernel from the sorted keys of the group shapes,
// which come first, in slot order (the longest items first).  starts /
// itemOff: the buckets' first keys and items; stripBytes: what their strips may
// take (0: none).
void makeUnits(const sqmi_sequences &V, Planned &P, const std::vector<size_t> &starts,
               const std::vector<size_t> &itemOff, int R16, int R64, double cellsStrip, int64_t stripBytes)
{
    const RawVec<Key> &keys = P.keys16;
    const size_t nb = starts.size() - 1;
    size_t bG = 0, b64 = 0;   // buckets of the group shapes, and of 64 lanes
    while (bG < nb && (keys[starts[bG]].key >> kKeyClassShift) < kSlotLane16) {
        if ((keys[starts[bG]].key >> kKeyClassShift) < kSlot16)
            b64 = bG + 1;
        ++bG;
    }
    const size_t nPairs = starts[bG], nItems = itemOff[bG], n64 = itemOff[b64];
    const bool par = (int64_t)nPairs > kParallelMin;
    P.order16.resize(nPairs);
#pragma omp parallel for schedule(static) if (par)
    for (int64_t k = 0; k < (int64_t)nPairs; ++k)
        P.order16[k] = keys[k].id;
    const int minBlocks = stripBytes <= 0 ? 0 : fixedShapeRule() && stripMinBlocks() < 0 ? 0 : stripMinBlocks();
    // An item as one unit, with its row units in `pad`.  Few pairs: the
    // units of its tallest pair (buckets may be coarse).
    auto item = [&](size_t b, size_t k, size_t e) {
        const uint32_t key = keys[starts[b]].key, slot = key >> kKeyClassShift;
        int64_t units = unitsOf(key);
        if (!par || slot < kSlot16) {
            int64_t maxM = 0;
            for (size_t x = k; x < e; ++x)
                maxM = std::max(maxM, V.offsets[keys[x].id + 1] - V.offsets[keys[x].id]);
            units = unitsOfRows(maxM);
        }
        return ScoreUnit{(int32_t)k, (int32_t)(e - k), widthOf(keys[k].key), 0, 0,
                         (slot < kSlot16 ? kUnit64 : 0) | (slot % 2 == 0 ? kUnitWide : 0), -1, (int32_t)units, 0};
    };
    // Rows: blocks of R rows per lane, block 0 as tall as needed.
    auto split = [](ScoreUnit &u, int R) {
        const int G = (u.shape & kUnit64) ? 64 : 16, rowsPerUnit = kUnitRows / G, per = R / rowsPerUnit;
        u.nblocks = (u.pad + per - 1) / per;
        int RH = (u.pad - per * (u.nblocks - 1)) * rowsPerUnit;
        if (G == 64 && RH > 4)   // compiled heights 1, 2, 3, 4, 6, 8, 12, 16
            RH = RH <= 6 ? 6 : RH <= 8 ? 8 : RH <= 12 ? 12 : 16;
        u.rows = R | std::min(RH, R) << 8;
    };
    auto padded = [](const ScoreUnit &u) -> int64_t {
        return (int64_t)2 * 64 * u.maxN * ((u.rows >> 8) + (int64_t)(u.nblocks - 1) * (u.rows & 0xff));
    };
    auto words = [](const ScoreUnit &u) -> int64_t { return ((u.shape & kUnit64) ? 1 : 4) * (int64_t)(u.maxN + 1); };
    auto strips = [&](const ScoreUnit &u) {
        if (u.nblocks < 2 || minBlocks == 0)
            return false;
        return minBlocks > 0 ? u.nblocks >= minBlocks
                             : (u.shape & kUnit64) && (double)u.maxN * u.pad * kUnitRows > cellsStrip;
    };
    auto addStrips = [&](ScoreUnit u) {
        u.rowOff = P.stripWords;
        P.stripWords += words(u) * u.nblocks;
        for (int b = 0; b < u.nblocks; ++b) {
            u.block = b;
            P.units.push_back(u);
        }
    };
    P.units.clear();
    P.items16 = (int64_t)nItems;

    // 64 lanes.  Strips of as few rows as give every resident wave about two.
    int stripR = R64 ? R64 : 4;
    if (!R64 && minBlocks < 0) {
        int64_t strips4 = 0;
        for (size_t b = 0; b < b64; ++b)
            strips4 += (int64_t)((starts[b + 1] - starts[b] + 1) / 2) * ((unitsOf(keys[starts[b]].key) + 3) / 4);
        while (stripR < 16 && strips4 * 4 / stripR > 2 * kResidentWaves)
            stripR *= 2;
    }
    P.units.reserve(nItems);
    std::vector<ScoreUnit> wave;
    wave.reserve(n64);
    const int64_t budget = stripBytes / 8;
    int64_t all = 0;   // words of every item that qualifies
    for (size_t b = 0; b < b64; ++b)
        for (size_t k = starts[b]; k < starts[b + 1]; k += 2) {
            ScoreUnit u = item(b, k, std::min(starts[b + 1], k + 2));
            split(u, R64 ? R64 : stripR);
            u.block = strips(u) ? 0 : -1;
            all += u.block < 0 ? 0 : words(u) * u.nblocks;
            wave.push_back(u);
        }
    // Past the budget: strips for the first items (the longest: a chain of its
    // own) and for the last ones (they level the waves' ends), the items in
    // between whole.  A quarter of the budget covers some hundred of the longest.
    if (all > budget) {
        int64_t used = 0;
        size_t from = 0, to = wave.size();
        auto take = [&](const ScoreUnit &u, int64_t limit) {
            const int64_t w = u.block < 0 ? 0 : words(u) * u.nblocks;
            const bool fits = used + w <= limit;
            used += fits ? w : 0;
            return fits;
        };
        while (from < to && take(wave[from], budget / 4))
            ++from;
        while (to > from && take(wave[to - 1], budget))
            --to;
        for (size_t k = from; k < to; ++k)
            wave[k].block = -1;
    }
    for (ScoreUnit &u : wave) {
        const bool s = u.block >= 0;
        u.block = -1;
        if (!s && !R64)
            split(u, 16);
        P.padded16 += padded(u);
        if (s) {
            addStrips(u);
        } else {
            P.slotWords = std::max(P.slotWords, words(u));
            P.units.push_back(u);
        }
    }
    // 16 lanes: whole items (strips on request only).
    if (minBlocks > 0) {
        for (size_t b = b64; b < bG; ++b)
            for (size_t k = starts[b]; k < starts[b + 1]; k += 8) {
                ScoreUnit u = item(b, k, std::min(starts[b + 1], k + 8));
                split(u, R16);
                P.padded16 += padded(u);
                if (strips(u) && P.stripWords + words(u) * u.nblocks <= budget) {
                    addStrips(u);
                } else {
                    P.slotWords = std::max(P.slotWords, words(u));
                    P.units.push_back(u);
                }
            }
        return;
    }
    const size_t at = P.units.size();
    P.units.resize(at + nItems - n64);
    int64_t slotWords = P.slotWords, pad = 0;
#pragma omp parallel for schedule(dynamic, 8) reduction(max : slotWords) reduction(+ : pad) if (par)
    for (int64_t b = (int64_t)b64; b < (int64_t)bG; ++b) {
        size_t it = at + itemOff[b] - n64;
        for (size_t k = starts[b]; k < starts[b + 1]; k += 8, ++it) {
            ScoreUnit u = item(b, k, std::min(starts[b + 1], k + 8));
            split(u, R16);
            slotWords = std::max(slotWords, words(u));
            pad += padded(u);
            P.units[it] = u;
        }
    }
    P.slotWords = slotWords;
    P.padded16 += pad;
}

// Routing (empty / int16 / int32) and length bucketing into work items.
// Pure host code: needs no device.  stripBytes: what strips may take (0: none).
// tight: the smallest lists, for a no-allocation call near its limit (16
// lanes per couple, every bin of the shape table's on lanes whatever its values).
void plan(const sqmi_sequences &H, const sqmi_sequences &V, const sqmi_scoring &scoring, uint32_t mode,
          uint32_t flags, Planned &P, bool traceShape = false, bool noLong = false, int64_t stripBytes = kMaxStripBytes,
          bool tight = false)
{
    P.flags = flags;
    const int64_t N = H.count;
    ScoringInfo &si = P.si;
    si.alpha = scoring.alphabet_size;
    si.o = scoring.gap_open;
    si.e = scoring.gap_extend;
    si.sMax = INT_MIN;
    si.sMin = INT_MAX;
    for (int k = 0; k < si.alpha * si.alpha; ++k) {
        si.sMax = std::max(si.sMax, scoring.table[k]);
        si.sMin = std::min(si.sMin, scoring.table[k]);
    }
    const bool local = (mode & SQMI_LOCAL) != 0;
    P.local = local;
    const bool costsOk16 = si.o <= 0 && si.e <= 0 && si.o >= -1024 && si.e >= -1024 && si.sMax <= 1024 &&
                           si.sMin >= -1024 && !(flags & SQMI_FORCE_INT32) &&
                           (si.alpha <= 4 || si.alpha + 1 <= kTabMaxCodes);
    // DNA byte profile: t(h, v) - gapOpen in 0..255.  Its padding column
    // (past n) is 0, i.e. t = gapOpen <= 0, so under local alignment the
    // cells past n stay at or below the maximum over columns 1..n, and an
    // equal one follows its source in column order.
    si.dna = si.alpha <= 4 && si.sMin - si.o >= 0 && si.sMax - si.o <= 255;
    si.dnaDrift = si.dna && si.sMax - si.o - std::max(si.o, si.e) <= 255;
    P.drift = driftOf(si, local);
    P.dna16 = local ? si.dna : si.dnaDrift;
    const Drift dr = P.drift;
    const bool dna16 = P.dna16;
    uint32_t track;
    if (local)
        track = kTrackLocal;
    else {
        track = 0;
        if (mode & SQMI_FREE_BOTTOM)
            track |= kTrackBottom;
        if (mode & SQMI_FREE_RIGHT)
            track |= kTrackRight;
        if (!track)
            track = kTrackEnd;
    }
    P.track = track;
    P.mode = mode;
    // Route every pair and give it a bucket key (see bucketOf).  The int16
    // pairs' shape slots: the trace shape, a forced shape, or lanes where the
    // table (wide global values: kWideLane) gives a pair's length bin to them,
    // else 16 or 64 lanes by its share of the call's cells (a pair that needs
    // more than 255 row blocks on lanes takes groups).
    RawVec<Key> &keys = P.keys16;
    keys.resize((size_t)N);
    int64_t cells = 0;
    // The long route: every AlignConfig and local for scores, global only
    // for the traceback.
    const bool allLong = longAll() && si.dna && (mode == 0 || !traceShape) && !noLong;
    const int64_t longMin0 = longMinSide();
    auto route16 = [&](int64_t n, int64_t m) {
        return !(allLong && n >= longMin0 && m >= longMin0) && costsOk16 && fitsInt16(si, n, m, local) &&
               n < (1 << kKeyNBits);
    };
    std::vector<Variant16> &shapes = P.shapes;
    shapes.clear();
    bool fineBin[16] = {};
    const int forcedG = (int)((flags >> 8) & 0xFF), forcedR = (int)((flags >> 16) & 0xFF);
    int R16 = 16, R64 = 0;          // rows per lane of the group shapes (R64 = 0: by the rule)
    int binLane[16] = {};           // one-pair-per-lane rows of a length bin, or 0
    int binG[16] = {};              // forced group size of a bin, or 0 (the rule)
    int wideLaneBin = -1;           // global pairs of wide values: the last bin on lanes (kWideLane)
    double cells64 = 0, cellsStrip = 0;
    if (traceShape) {
        shapes.push_back(Variant16{kTraceLanes, kTraceRows / kTraceLanes, dna16, track});
    } else {
        for (int w = 1; w >= 0; --w)
            shapes.push_back(Variant16{64, 16, dna16, track, w != 0});
        for (int w = 1; w >= 0; --w)
            shapes.push_back(Variant16{16, 16, dna16, track, w != 0});
        shapes.push_back(Variant16{1, 16, dna16, track});
        shapes.push_back(Variant16{1, 32, dna16, track});
        shapes.push_back(Variant16{1, forcedG == 1 ? forcedR : 32, dna16, track, true});
        // Pairs per length bin and cells of the int16 route; global pairs of
        // wide values where there may be enough of them for lanes.
        int64_t binCount[16] = {}, binWide[16] = {}, cells16 = 0, most16 = 0;
        const bool countWide = !local && N >= kWideLane[3].alone;
#pragma omp parallel if (N > kParallelMin)
        {
            int64_t local16[16] = {}, localWide[16] = {}, localCells = 0, localMost = 0;
#pragma omp for schedule(static) nowait
            for (int64_t i = 0; i < N; ++i) {
                const int64_t n = H.offsets[i + 1] - H.offsets[i];
                const int64_t m = V.offsets[i + 1] - V.offsets[i];
                if (n != 0 && m != 0 && route16(n, m)) {
                    const int b = lengthBin(m);
                    ++local16[b];
                    if (countWide && b <= kWideLane[0].bin)
                        localWide[b] += !driftNarrow(si, dr, local, n, m);
                    localCells += n * m;
                    localMost = std::max(localMost, n * m);
                }
            }
#pragma omp critical
            {
                for (int b = 0; b < 16; ++b) {
                    binCount[b] += local16[b];
                    binWide[b] += localWide[b];
                }
                cells16 += localCells;
                most16 = std::max(most16, localMost);
            }
        }
        int64_t pairs16 = 0;
        for (int b = 0; b < 16; ++b)
            pairs16 += binCount[b];
        cells64 = kCouple64Share * (double)cells16;
        cellsStrip = kStripShare * (double)cells16;
        if ((double)most16 * (double)pairs16 <= 4.0 * (double)cells16 && evenOn16((double)most16, (double)pairs16, (double)cells16, dna16))
            cells64 = cellsStrip = 1e300;
        if (tight)
            cells64 = 1e300;
        if (fixedShapeRule()) {
            std::fill(binG, binG + 16, 16);
        } else {
            for (int b = 0; b < 16; ++b)
                binLane[b] = laneRows(shapeCategory(dna16, local), b, pairs16);
            for (const WideLane &q : kWideLane) {
                int64_t below = 0;
                for (int b = 0; b <= q.bin; ++b)
                    below += binWide[b];
                if (countWide && wideLaneBin < 0 && below >= (below == pairs16 ? q.alone : q.beside))
                    wideLaneBin = q.bin;
            }
        }
        // SQMI_BIN_SHAPES="b:G:R,...": the form of bin b in place of the
        // table's (the tuner times calls with it): 1:R one pair per lane, 0:0
        // groups by the rule, or a group shape, whose rows R then hold for
        // every bin of that group size (units have one row count each); forced
        // shapes: every bin's.
        auto force = [&](int b, int g, int r) {
            if (g == 0 && r == 0)
                binG[b] = binLane[b] = 0;
            if (!shapeSupported(Variant16{g, r, dna16, track}))
                return;
            binG[b] = g == 1 ? 0 : g;
            binLane[b] = g == 1 ? r : 0;
            if (g == 16)
                R16 = r;
            if (g == 64)
                R64 = r;
        };
        if (const char *env = std::getenv("SQMI_BIN_SHAPES")) {
            for (const char *c = env; *c;) {
                int b = -1, g = 0, r = 0, used = 0;
                if (std::sscanf(c, "%d:%d:%d%n", &b, &g, &r, &used) != 3)
                    break;
                if (b >= 0 && b < 16)
                    force(b, g, r);
                c += used;
                if (*c == ',')
                    ++c;
            }
        }
        if (forcedG && forcedR)
            for (int b = 0; b < 16; ++b)
                force(b, forcedG, forcedR);
        const int unitsMode = rowUnitsMode();
        for (int b = 0; b < 16; ++b)
            fineBin[b] = unitsMode == 2 || (unitsMode == 0 && binCount[b] >= kFineUnitPairs);
    }
    // Shape slot and row units of an int16 pair.
    auto slotOf = [&](int64_t n, int64_t m, int64_t &units) -> uint32_t {
        if (traceShape) {
            units = blocksFor(shapes[0], m);
            return 0;
        }
        const int b = lengthBin(m);
        const bool wide = !driftNarrow(si, dr, local, n, m);
        if (local || !wide || forcedG == 1 || tight ? binLane[b] != 0 : b <= wideLaneBin && !binG[b]) {
            const uint32_t slot = !local && wide ? kSlotLaneWide : binLane[b] == 32 ? kSlotLane32 : kSlotLane16;
            units = blocksFor(shapes[slot], m);
            if (units <= kMaxBlocks16)
                return slot;
        }
        const bool g64 = binG[b] ? binG[b] == 64 : (double)n * (double)m > cells64;
        units = unitsOfRows(m);
        if (!fineBin[b]) {
            // Pairs of an item have their row 0 in block 0: coarse units span
            // no more than a block (R = 8 on 16 lanes: 128 rows).
            const int64_t per = !g64 && R16 == 8 ? 2 : 4;
            units = (units + per - 1) / per * per;
        }
        return (g64 ? kSlot64 : kSlot16) + (wide ? 0u : 1u);
    };
#pragma omp parallel for schedule(static) reduction(+ : cells) if (N > kParallelMin)
    for (int64_t i = 0; i < N; ++i) {
        const int64_t n = H.offsets[i + 1] - H.offsets[i];
        const int64_t m = V.offsets[i + 1] - V.offsets[i];
        uint32_t key = kClassRest << kKeyClassShift;
        if (n != 0 && m != 0) {
            cells += n * m;
            if (route16(n, m)) {
                int64_t units = 0;
                const uint32_t slot = slotOf(n, m, units);
                if (units <= 1023 && !(traceShape && units > kMaxBlocks16))
                    key = (slot << kKeyClassShift) | ((1023u - (uint32_t)units) << kKeyNBits) |
                          ((1u << kKeyNBits) - 1 - (uint32_t)n);
            }
        }
        keys[i] = Key{key, (int32_t)i};
    }
    P.cells = cells;
    radixSort(keys, P.keysTmp, P.sortHist);
    // Segments of the sorted order: int16 (by shape), then int32 and empty.
    size_t n16 = 0;
    while (n16 < keys.size() && (keys[n16].key >> kKeyClassShift) < kClassRest) {
        // Jump by bucket boundaries found with a binary search.
        const uint32_t cls = keys[n16].key >> kKeyClassShift;
        n16 = (size_t)(std::upper_bound(keys.begin() + n16, keys.end(), ((cls + 1) << kKeyClassShift) - 1,
                                        [](uint32_t v, const Key &k) { return v < k.key; }) -
                       keys.begin());
    }
    const int64_t longMin = longMinSide();
    const bool longOk = si.dna && (mode == 0 || !traceShape) && !noLong;
    for (size_t k = n16; k < keys.size(); ++k) {
        const int32_t i = keys[k].id;
        const int64_t n = H.offsets[i + 1] - H.offsets[i];
        const int64_t m = V.offsets[i + 1] - V.offsets[i];
        if (n == 0 || m == 0) {
            P.emptyIds.push_back(i);
            continue;
        }
        if (longOk && n >= longMin && m >= longMin && fitsLong32(si, n, m)) {
            P.idsLong.push_back(i);
            continue;
        }
        P.ids32.push_back(i);
        P.scratchOff32.push_back(P.scratch32);
        // score: H and E columns (int32 pairs); traceback: the columns plus
        // one trace byte per cell, 16-byte aligned.
        P.scratch32 += traceShape ? ((8 * (m + 1) + (n + 1) * (m + 1) + 15) & ~(int64_t)15) : m + 1;
    }
    keys.resize(n16);
    RawVec<Key> &keys16 = P.keys16;

    // Work items: each bucket (shape, row blocks) is cut into runs of up to
    // pairs-per-wave pairs, in sorted order.  Bucket starts are found in
    // parallel, then every bucket writes its own items.
    std::vector<size_t> starts;
    {
        int T = 1;
#ifdef _OPENMP
        T = std::max(1, std::min(omp_get_max_threads(), (int)(n16 / 16384) + 1));
#endif
        std::vector<std::vector<size_t>> part((size_t)T);
#pragma omp parallel num_threads(T)
        {
            int t = 0;
#ifdef _OPENMP
            t = omp_get_thread_num();
#endif
            const size_t lo = n16 * t / T, hi = n16 * (t + 1) / T;
            for (size_t k = lo; k < hi; ++k)
                if (k == 0 || bucketOf(keys16[k].key) != bucketOf(keys16[k - 1].key))
                    part[t].push_back(k);
        }
        for (auto &v : part)
            starts.insert(starts.end(), v.begin(), v.end());
        starts.push_back(n16);
    }
    const size_t nb = starts.size() - 1;
    std::vector<size_t> itemOff(nb + 1, 0);
    for (size_t b = 0; b < nb; ++b) {
        const int PP = pairsPerWave(shapes[keys16[starts[b]].key >> kKeyClassShift]);
        itemOff[b + 1] = itemOff[b] + (starts[b + 1] - starts[b] + PP - 1) / PP;
    }
    std::vector<Plan16> &plans = P.plans;
    if (!traceShape)
        makeUnits(V, P, starts, itemOff, R16, R64, cellsStrip, stripBytes);
    for (uint32_t v = traceShape ? 0 : kSlotLane16; v < (uint32_t)shapes.size(); ++v) {
        // The shape's contiguous range of buckets and of sorted pairs.
        size_t b0 = 0;
        while (b0 < nb && (keys16[starts[b0]].key >> kKeyClassShift) < v)
            ++b0;
        size_t b1 = b0;
        while (b1 < nb && (keys16[starts[b1]].key >> kKeyClassShift) == v)
            ++b1;
        if (b0 == b1)
            continue;
        plans.push_back(Plan16{});
        Plan16 &pl = plans.back();
        pl.var = shapes[v];
        const size_t p0 = starts[b0], p1 = starts[b1];
        const size_t i0 = itemOff[b0];
        const int PP = pairsPerWave(pl.var);
        pl.order.resize(p1 - p0);
        pl.items.resize(itemOff[b1] - i0);
        int32_t maxN = 0;
#pragma omp parallel for schedule(static) reduction(max : maxN) if (p1 - p0 > (size_t)kParallelMin)
        for (int64_t k = (int64_t)p0; k < (int64_t)p1; ++k) {
            pl.order[k - p0] = keys16[k].id;
            maxN = std::max(maxN, widthOf(keys16[k].key));
        }
        pl.maxN = maxN;
#pragma omp parallel for schedule(dynamic, 8) if (p1 - p0 > (size_t)kParallelMin)
        for (int64_t b = (int64_t)b0; b < (int64_t)b1; ++b) {
            size_t it = itemOff[b] - i0;
            const int32_t nblocks = unitsOf(keys16[starts[b]].key);
            for (size_t k = starts[b]; k < starts[b + 1]; k += PP, ++it) {
                const size_t e = std::min(starts[b + 1], k + PP);
                // Widest first inside a bucket: the first pair has the item's width.
                pl.items[it] = WorkItem{(int32_t)(k - p0), (int32_t)(e - k), widthOf(keys16[k].key), nblocks};
            }
        }
    }
}

void fillStats(const Planned &P, sqmi_stats &st)
{
    st.pairs = (int64_t)(P.emptyIds.size() + P.ids32.size() + P.idsLong.size() + P.keys16.size());
    st.cells = P.cells;
    st.pairs_int32 = (int64_t)(P.ids32.size() + P.idsLong.size());
    st.pairs_long = (int64_t)P.idsLong.size();
    st.pairs_long_packed = (longPacked(P.si, P.flags) && P.mode == 0) ? st.pairs_long : 0;
    st.pairs_int16 = (int64_t)P.keys16.size();
    int64_t items = P.items16, padded = P.padded16;
    st.pairs_lane = 0;
    for (const Plan16 &pl : P.plans) {
        items += (int64_t)pl.items.size();
        if (pl.var.G == 1)
            st.pairs_lane += (int64_t)pl.order.size();
        for (const WorkItem &w : pl.items)
            padded += 2LL * (64 / pl.var.G) * (int64_t)w.maxN * w.nblocks * pl.var.G * pl.var.R;
    }
    st.work_items = items;
    st.padded_cells = padded;
}

// An item of the trace kernel: up to 128 / lanes pairs of `nblocks` blocks.
struct TraceItem {
    int32_t first, count, maxN, nblocks, lanes;
};
// 1 KB records of an item (a step of four couples on 16 lanes, four steps of one on 64).
int64_t traceRecsOf(const TraceItem &w)
{
    const int64_t steps = (int64_t)w.nblocks * traceSteps(w.maxN, w.lanes);
    return w.lanes == 64 ? (steps + 3) / 4 : steps;
}

// Lanes per couple of the trace kernel, by the time an item takes against the
// whole call's.  On 16 lanes a step takes a wave 0.53 us (0.47 of a full
// SIMD) and a block starts about 110 steps behind the one above; on 64 lanes of 4
// rows 0.2 us for a quarter of the couples, which costs 1.4 times as much.
// So items go to 64 lanes whose chain of blocks would take more than a share
// of the call's time on a full chip (with the table, whose lookups weigh more
// there, a larger one).  SQMI_TRACE_LANES=16 or 64 takes one form for all
// (tests).  Device time of 8,191 uneven DNA pairs, shares 0.5 / 1 / 2 / 4: 4.3 /
// 4.7 / 5.5 / 8.7 ms (all on 64 lanes 4.4, on 16 8.6); of 8,192 protein pairs,
// local: 4.3 / 3.5 / 3.6 / 3.5 (4.2, 3.5); 65,536 pairs of 1 kbp: none, 17.4
// (all on 64 lanes 20.2).
constexpr double kTrace64Share = 0.5, kTrace64ShareTab = 1.5;
void traceItems(const sqmi_sequences &H, const Plan16 &pl, bool dna, std::vector<TraceItem> &out)
{
    double total = 0;
    for (const WorkItem &w : pl.items)
        total += (double)w.nblocks * traceSteps(w.maxN, 16) * 0.47 / 1024;
    const char *env = std::getenv("SQMI_TRACE_LANES");
    const int forced = env && *env ? std::atoi(env) : 0;
    out.clear();
    out.reserve(pl.items.size());
    for (const WorkItem &w : pl.items) {
        const double chain = (w.maxN + 110.0 * w.nblocks) * 0.53;
        if (forced == 16 || (forced != 64 && chain <= (dna ? kTrace64Share : kTrace64ShareTab) * total)) {
            out.push_back(TraceItem{w.first, w.count, w.maxN, w.nblocks, 16});
            continue;
        }
        for (int32_t f = w.first; f < w.first + w.count; f += 2) {
            TraceItem q{f, std::min<int32_t>(2, w.first + w.count - f), 1, w.nblocks, 64};
            for (int32_t x = f; x < f + q.count; ++x)
                q.maxN = std::max(q.maxN, (int32_t)(H.offsets[pl.order[x] + 1] - H.offsets[pl.order[x]]));
            out.push_back(q);
        }
    }
}

sqmi_status validate(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                     const sqmi_scoring *scoring, uint32_t &mode)
{
    sqmi_status st;
    if ((st = checkSet(ctx, setH, "set_h")) != SQMI_OK || (st = checkSet(ctx, setV, "set_v")) != SQMI_OK)
        return st;
    if (setH->count != setV->count)
        return fail(ctx, SQMI_ERR_LENGTH_MISMATCH, "set_h and set_v differ in length");
    if (!scoring || !scoring->table || scoring->alphabet_size < 1 || scoring->alphabet_size > 32)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "scoring: alphabet_size must be 1..32 with a table");
    if (mode & ~31u)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "mode: unknown bits");
    if (mode & SQMI_LOCAL)
        mode = SQMI_LOCAL;   // localAlignmentScore has no AlignConfig
    return SQMI_OK;
}

sqmi_status checkForced(sqmi_context *ctx, uint32_t flags)
{
    const int g = (int)((flags >> 8) & 0xFF), r = (int)((flags >> 16) & 0xFF);
    if (!g && !r)
        return SQMI_OK;
    for (bool dna : {true, false})
        if (!shapeSupported(Variant16{g, r, dna, kTrackEnd}))
            return fail(ctx, SQMI_ERR_UNSUPPORTED, "forced kernel variant is not compiled");
    return SQMI_OK;
}


// Bytes the traceback may hold in trace records or int32 trace scratch at
// once: a quarter of the device's memory, at least 8 GiB and at most 64 GiB
// (72 GB -> 64 GiB on a 288 GB MI355X), or SQMI_TRACE_BUDGET_MB from the
// environment.
int64_t traceBudget(const sqmi_context *ctx)
{
    const char *env = std::getenv("SQMI_TRACE_BUDGET_MB");
    if (env && *env) {
        const long long mb = std::atoll(env);
        if (mb > 0)
            return (int64_t)mb << 20;
    }
    const int64_t quarter = ctx ? ctx->totalMem / 4 : 0;
    return std::min<int64_t>(std::max<int64_t>(quarter, (int64_t)8 << 30), (int64_t)64 << 30);
}

// Device copies of what every entry point needs: residues (unless already on
// the device), offsets, the output scores buffer (unless the caller's is on
// the device) and the substitution tables: t(h, v) = s(h, v) - gapOpen with a
// padding code (int16 kernels), its byte profile (DNA path) and the plain
// table (int32 kernels).  The host staging data of the asynchronous copies
// lives in the struct, which the caller keeps until its stream is synchronised.
struct Inputs
{
    const uint8_t *dH = nullptr, *dV = nullptr;
    int32_t *dScores = nullptr;
    std::vector<int16_t> tTab;
    // DNA profiles: dwords 0..7 by column residue h (byte v = t(h, v)),
    // dwords 8..15 by row residue v (byte h = t(h, v)); the padding code
    // (alpha) maps to zero bytes.
    uint32_t prof[16] = {};
};

// Residue sets of up to this many bytes go through the stage.
constexpr int64_t kStageResidues = (int64_t)1 << 20;

// Bytes uploadInputs() puts into the stage, at most.
size_t stageInputs(const sqmi_sequences *setH, const sqmi_sequences *setV, const sqmi_scoring *scoring, uint32_t flags)
{
    const int64_t N = setH->count, A = scoring->alphabet_size;
    size_t bytes = 2 * stageBytes(8 * (N + 1)) + stageBytes(2 * (A + 1) * (A + 1)) + stageBytes(64) + stageBytes(4 * A * A);
    if (!(flags & SQMI_RESIDUES_ON_DEVICE) && setH->offsets[N] + setV->offsets[N] <= kStageResidues)
        bytes += stageBytes(setH->offsets[N]) + stageBytes(setV->offsets[N]) + 512;
    return bytes;
}

size_t downScores(int64_t N, uint32_t flags) { return flags & SQMI_SCORES_ON_DEVICE ? 0 : stageBytes(4 * (size_t)N); }

// A host thread that is joined when it goes out of scope (early returns
// included).
struct JoinedThread {
    std::thread t;
    ~JoinedThread()
    {
        if (t.joinable())
            t.join();
    }
    void join()
    {
        if (t.joinable())
            t.join();
    }
};

// Host residues into the context's buffers (in.dH / in.dV).
hipError_t uploadResidues(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV, Inputs &in)
{
    const int64_t N = setH->count;
    const int64_t hTot = setH->offsets[N], vTot = setV->offsets[N];
    hipError_t err;
    if (hTot + vTot <= kStageResidues && stageFits(ctx, stageBytes(hTot) + stageBytes(vTot) + 512)) {
        // (256 bytes of slack after the residues, 64 below.)
        if ((err = put(ctx, ctx->b.hRes, setH->residues, hTot)) != hipSuccess)
            return err;
        ctx->pinUsed += 256;
        if ((err = put(ctx, ctx->b.vRes, setV->residues, vTot)) != hipSuccess)
            return err;
        ctx->pinUsed += 256;
    } else if ((err = ensure(ctx->b.hRes, hTot + 64)) != hipSuccess || (err = ensure(ctx->b.vRes, vTot + 64)) != hipSuccess ||
        (err = hipMemcpyAsync(ctx->b.hRes.p, setH->residues, hTot, hipMemcpyHostToDevice, ctx->stream)) !=
            hipSuccess ||
        (err = hipMemcpyAsync(ctx->b.vRes.p, setV->residues, vTot, hipMemcpyHostToDevice, ctx->stream)) != hipSuccess)
        return err;
    in.dH = static_cast<const uint8_t *>(ctx->b.hRes.p);
    in.dV = static_cast<const uint8_t *>(ctx->b.vRes.p);
    return hipSuccess;
}

// Residues (unless uploadResidues already ran for `in`), offsets, tables.
sqmi_status uploadInputs(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                         const sqmi_scoring *scoring, const ScoringInfo &si, int32_t *scores, uint32_t flags,
                         Inputs &in)
{
    const int64_t N = setH->count;
    hipError_t err;
    const uint8_t *dH = setH->residues, *dV = setV->residues;
    if (!(flags & SQMI_RESIDUES_ON_DEVICE)) {
        if (!in.dH && (err = uploadResidues(ctx, setH, setV, in)) != hipSuccess)
            return hipFail(ctx, err, "copying residues");
        dH = in.dH;
        dV = in.dV;
    }
    if ((err = put(ctx, ctx->b.hOff, setH->offsets, 8 * (N + 1))) != hipSuccess ||
        (err = put(ctx, ctx->b.vOff, setV->offsets, 8 * (N + 1))) != hipSuccess)
        return hipFail(ctx, err, "copying offsets");
    int32_t *dScores = scores;
    if (!(flags & SQMI_SCORES_ON_DEVICE)) {
        if ((err = ensure(ctx->b.scores, 4 * N)) != hipSuccess)
            return hipFail(ctx, err, "allocating scores");
        dScores = static_cast<int32_t *>(ctx->b.scores.p);
    }

    // Substitution tables: t(h, v) = s(h, v) - gapOpen with a padding code.
    const int A = si.alpha, TW = A + 1;
    std::vector<int16_t> &tTab = in.tTab;
    tTab.assign((size_t)TW * TW, -1024);
    for (int h = 0; h < A; ++h)
        for (int v = 0; v < A; ++v)
            tTab[h * TW + v] = (int16_t)(scoring->table[h * A + v] - si.o);
    uint32_t *prof = in.prof;
    if (si.dna)
        for (int h = 0; h < A; ++h)
            for (int v = 0; v < A; ++v) {
                prof[h] |= (uint32_t)(scoring->table[h * A + v] - si.o) << (8 * v);
                prof[8 + v] |= (uint32_t)(scoring->table[h * A + v] - si.o) << (8 * h);
            }
    if ((err = put(ctx, ctx->b.tTable, tTab.data(), tTab.size() * 2)) != hipSuccess ||
        (err = put(ctx, ctx->b.dnaProf, prof, 64)) != hipSuccess ||
        (err = put(ctx, ctx->b.table32, scoring->table, 4 * A * A)) != hipSuccess)
        return hipFail(ctx, err, "copying tables");
    in.dH = dH;
    in.dV = dV;
    in.dScores = dScores;
    return SQMI_OK;
}

// Device addresses of the alignment rows output (all null: no rows).
struct RowsDev {
    uint8_t *ops = nullptr;
    const int64_t *opOff = nullptr;
    int64_t *opLen = nullptr;
    int64_t *begins = nullptr;   // local windows only
};

// Host copies of the long pairs' descriptors (kept until the caller has
// synchronised).
struct LongStage {
    std::vector<LongPair> pairs;
    std::vector<LongCouple> couples;
    std::vector<int2> units;
};

// The packed kernels' long pairs (`ids`, longest first, so that couples hold
// similar shapes), in chunks of couples whose buffers fit traceBudget().
sqmi_status runLong16(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV, const Planned &P,
                      const Inputs &in, int32_t *dCounts, const RowsDev &rows, const std::vector<int32_t> &ids,
                      LongStage &stage, Deferred *deferred)
{
    hipStream_t stream = ctx->stream;
    const int64_t budget = traceBudget(ctx), N = setH->count;
    const size_t nc = (ids.size() + 1) / 2;
    auto sides = [&](size_t k, int32_t &n, int32_t &m) {
        n = (int32_t)(setH->offsets[ids[k] + 1] - setH->offsets[ids[k]]);
        m = (int32_t)(setV->offsets[ids[k] + 1] - setV->offsets[ids[k]]);
    };
    // Rows per lane by the time the call should take.  A step of a strip of 4,
    // 8 or 16 rows per lane takes a wave alone on its SIMD 115, 153 or 230
    // ns, and 63, 111 or 203 ns of a full one's; a strip starts about 160
    // steps behind the one above.  Either the chain of one couple's strips
    // bounds the call or the rounds of strips on the chip's SIMDs do, plus
    // their start.  Forward of 100 kbp pairs, R = 8 / 16: 10 pairs 20.1 / 27
    // ms, 20: 28.3 / 27.2, 40: 45.5 / 43.6, 64: 68 / 77 (a fourth round
    // for 64 strips).  SQMI_LONG_ROWS sets R for tests.
    int R = 4;
    double best = 0;
    for (const LongCost &q : kLongCosts) {
        double strips = 0, chain = 0, lead = 0, steps = 0;
        for (size_t k = 0; k < ids.size(); k += 2) {
            int32_t n, m, n1 = 0, m1 = 0;
            sides(k, n, m);
            if (k + 1 < ids.size())
                sides(k + 1, n1, m1);
            const double nb = std::max(m, m1) / (64 * q.rows) + 1, len = std::max(n, n1);
            strips += nb;
            steps += nb * len;
            lead = std::max(lead, 160 * nb * q.alone);
            chain = std::max(chain, (len + 160 * nb) * q.alone);
        }
        const double rounds = strips / (4 * std::max(1, ctx->numCUs));
        const double t = std::max(chain, std::ceil(rounds) * (steps / strips) * q.full + lead);
        if (longRowsFit(P.si, q.rows) && (best == 0 || t < best)) {
            best = t;
            R = q.rows;
        }
    }
    if (const char *env = std::getenv("SQMI_LONG_ROWS")) {
        const int r = std::atoi(env);
        if ((r == 4 || r == 8 || r == 16) && longRowsFit(P.si, r))
            R = r;
    }
    std::vector<LongCouple> &couples = stage.couples;
    couples.assign(nc, LongCouple{});
    std::vector<size_t> chunkEnd, unitEnd;
    int64_t rowWords = 0, stateWords = 0, bytes = 0, maxRows = 1, maxState = 0;
    const int64_t traceBytes = dCounts ? (int64_t)2 * longWinStrips(R) * kWinCouples * kLongT * 64 * longRecBytes(R) : 0;
    size_t maxCouples = 1, first = 0;
    for (size_t c = 0; c < nc; ++c) {
        LongCouple &q = couples[c];
        for (int x = 0; x < 2; ++x) {
            const size_t k = 2 * c + x;
            q.pid[x] = -1;
            if (k < ids.size()) {
                q.pid[x] = ids[k];
                sides(k, q.n[x], q.m[x]);
            }
        }
        q.maxN = std::max(q.n[0], q.n[1]);
        q.nb = std::max(q.m[0], q.m[1]) / (64 * R) + 1;
        for (int x = 0; x < 2; ++x)
            q.p[x] = q.nb * 64 * R - 1 - q.m[x];
        q.chunks = (longSteps(q.maxN) + kLongT - 1) / kLongT;
        const int64_t rw = (int64_t)(q.nb - 1) * (q.maxN + 1);
        const int64_t sw = dCounts ? (int64_t)q.nb * q.chunks * longStateWords(R) * 64 : 0;
        const int64_t need = 8 * rw + 4 * sw + traceBytes;
        if (bytes > 0 && bytes + need > budget) {
            chunkEnd.push_back(c);
            first = c;
            rowWords = stateWords = bytes = 0;
        }
        q.rows = rowWords;
        q.state = stateWords;
        rowWords += rw;
        stateWords += sw;
        bytes += need;
        maxRows = std::max(maxRows, rowWords);
        maxState = std::max(maxState, stateWords);
        maxCouples = std::max(maxCouples, c + 1 - first);
    }
    chunkEnd.push_back(nc);
    std::vector<int2> &units = stage.units;
    units.clear();
    size_t b = 0;
    for (size_t e : chunkEnd) {
        int nb = 0;
        for (size_t c = b; c < e; ++c)
            nb = std::max(nb, couples[c].nb);
        for (int s = 0; s < nb; ++s)
            for (size_t c = b; c < e; ++c)
                if (s < couples[c].nb)
                    units.push_back(make_int2((int)(c - b), s));
        unitEnd.push_back(units.size());
        b = e;
    }
    if (units.size() >= (size_t)INT32_MAX)
        return fail(ctx, SQMI_ERR_UNSUPPORTED, "long pairs: too many strips for one launch");
    hipError_t err;
    const size_t qWords = 16 * chunkEnd.size();
    // (Bottom rows apart from the score and trace kernels' strips: the same
    // call's launches may hold those by address already.)
    if ((err = ensure(ctx->b.longRows, (size_t)maxRows * 8)) != hipSuccess ||
        (err = ensure(ctx->b.longPairs, sizeof(LongCouple) * nc)) != hipSuccess ||
        (err = ensure(ctx->b.longSched, 4 * qWords + sizeof(int2) * units.size())) != hipSuccess ||
        (err = ensure(ctx->b.endEF, (size_t)8 * N)) != hipSuccess)
        return hipFail(ctx, err, "allocating long-pair buffers");
    if (dCounts && ((err = ensure(ctx->b.longCk, (size_t)maxState * 4)) != hipSuccess ||
                    (err = ensure(ctx->b.longWalk, (size_t)8 * kLongWalkInts * maxCouples)) != hipSuccess ||
                    (err = ensure(ctx->b.longTrace, (size_t)traceBytes * maxCouples)) != hipSuccess))
        return hipFail(ctx, err, "allocating long-pair traceback buffers");
    uint32_t *queues = static_cast<uint32_t *>(ctx->b.longSched.p);
    int2 *dUnits = reinterpret_cast<int2 *>(queues + qWords);
    if ((err = hipMemcpyAsync(ctx->b.longPairs.p, couples.data(), sizeof(LongCouple) * nc, hipMemcpyHostToDevice, stream)) !=
            hipSuccess ||
        (err = hipMemcpyAsync(dUnits, units.data(), sizeof(int2) * units.size(), hipMemcpyHostToDevice, stream)) != hipSuccess)
        return hipFail(ctx, err, "uploading long pairs");
    hipError_t opErr = hipSuccess;
    auto op = [&](std::function<hipError_t()> f) {
        if (deferred)
            deferred->push_back(std::move(f));
        else if (opErr == hipSuccess)
            opErr = f();
        return opErr;
    };
    if ((err = op([=] { return launchZero32(queues, qWords, stream); })) != hipSuccess)
        return hipFail(ctx, err, "launching queue reset");
    b = 0;
    size_t ub = 0;
    for (size_t k = 0; k < chunkEnd.size(); ++k) {
        const size_t e = chunkEnd[k], ue = unitEnd[k];
        LongArgs a{};
        a.hRes = in.dH;
        a.vRes = in.dV;
        a.hOff = static_cast<const int64_t *>(ctx->b.hOff.p);
        a.vOff = static_cast<const int64_t *>(ctx->b.vOff.p);
        a.couples = static_cast<const LongCouple *>(ctx->b.longPairs.p) + b;
        a.nCouples = (int32_t)(e - b);
        a.units = dUnits + ub;
        a.nUnits = (int32_t)(ue - ub);
        a.queue = queues + 16 * k;
        a.rows = static_cast<uint64_t *>(ctx->b.longRows.p);
        a.state = dCounts ? static_cast<uint32_t *>(ctx->b.longCk.p) : nullptr;
        a.error = ctx->waitFlag;
        a.target = longTarget(P.si, P.drift);
        a.alpha = P.si.alpha;
        a.dnaProfile = static_cast<const uint32_t *>(ctx->b.dnaProf.p);
        a.drift = P.drift;
        a.scores = in.dScores;
        a.endEF = static_cast<int32_t *>(ctx->b.endEF.p);
        int64_t words = 0, maxM = 0, maxN = 0;
        for (size_t c = b; c < e; ++c) {
            words = std::max(words, couples[c].rows + (int64_t)(couples[c].nb - 1) * (couples[c].maxN + 1));
            maxM = std::max<int64_t>(maxM, std::max(couples[c].m[0], couples[c].m[1]));
            maxN = std::max<int64_t>(maxN, couples[c].maxN);
        }
        const int numCUs = std::max(1, ctx->numCUs);
        if ((err = op([=] {
                 const hipError_t z = launchZero32(reinterpret_cast<uint32_t *>(a.rows), 2 * (size_t)words, stream);
                 return z != hipSuccess ? z : launchLong16(R, a, numCUs, stream);
             })) != hipSuccess)
            return hipFail(ctx, err, "launching long-pair forward");
        if (dCounts) {
            a.trace = ctx->b.longTrace.p;
            a.walk = static_cast<int32_t *>(ctx->b.longWalk.p);
            a.counts = dCounts;
            a.linear = P.si.o == P.si.e;
            a.alwaysOpen = P.si.e < P.si.o;
            a.ops = rows.ops;
            a.opOff = rows.opOff;
            a.opLen = rows.opLen;
            if ((err = op([=] { return launchLong16WalkInit(a, stream); })) != hipSuccess)
                return hipFail(ctx, err, "launching long-pair walk init");
            // A round leaves its window through the top (at least winStrips
            // - 1 strips up) or the left side (all its chunks but one, less
            // the 63 columns between a strip's first and last lane).
            const int64_t up = (int64_t)(longWinStrips(R) - 1) * 64 * R, left = (kWinChunks - 1) * kLongT - 63;
            const int64_t rounds = (maxM + up - 1) / up + (maxN + left - 1) / left + 2;
            for (int64_t r = 0; r < rounds; ++r)
                if ((err = op([=] { return launchLong16Round(R, a, stream); })) != hipSuccess)
                    return hipFail(ctx, err, "launching long-pair traceback");
        }
        b = e;
        ub = ue;
    }
    return SQMI_OK;
}

// Long pairs: the packed kernels (runLong16) where the scoring allows and the
// alignment is global, else the tiled int32 forward (one launch per tile
// anti-diagonal), then, with `dCounts`, the checkpointed traceback: per round
// every unfinished pair's current window is recomputed with trace records and
// walked.  Pairs run in chunks whose checkpoints fit traceBudget().  `stage`
// holds the host copies of the descriptors until the caller synchronises.
sqmi_status runLong(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV, const Planned &P,
                    const Inputs &in, uint32_t flags, int32_t *dCounts, const RowsDev &rows,
                    LongStage &stage, Deferred *deferred = nullptr)
{
    std::vector<LongPair> &pairs = stage.pairs;
    // Stream operations run at once, or are appended to `deferred` (all
    // uploads and allocations still happen here).
    hipError_t opErr = hipSuccess;
    auto op = [&](std::function<hipError_t()> f) {
        if (deferred)
            deferred->push_back(std::move(f));
        else if (opErr == hipSuccess)
            opErr = f();
        return opErr;
    };
    if (P.idsLong.empty())
        return SQMI_OK;
    hipStream_t stream = ctx->stream;
    const int C = kLongTileC;
    const int64_t budget = traceBudget(ctx);
    const int64_t N = setH->count;
    // The packed kernels are global only; free end gaps and local take the
    // int32 forward and a result pass over its checkpoints.
    // Longest first, so that the couples of the packed kernels pair similar shapes.
    std::vector<int32_t> ids(P.idsLong);
    std::stable_sort(ids.begin(), ids.end(), [&](int32_t x, int32_t y) {
        const int64_t mx = setV->offsets[x + 1] - setV->offsets[x], my = setV->offsets[y + 1] - setV->offsets[y];
        const int64_t nx = setH->offsets[x + 1] - setH->offsets[x], ny = setH->offsets[y + 1] - setH->offsets[y];
        return mx != my ? mx > my : nx > ny;
    });
    if (longPacked(P.si, flags) && P.mode == 0)
        return runLong16(ctx, setH, setV, P, in, dCounts, rows, ids, stage, deferred);
    // Descriptors with checkpoint offsets relative to the pair's chunk.
    std::vector<size_t> chunkEnd;
    int64_t run = 0, maxRun = 0, bestRun = 0;
    pairs.clear();
    for (int32_t id : ids) {
        LongPair lp{};
        lp.pid = id;
        lp.n = (int32_t)(setH->offsets[id + 1] - setH->offsets[id]);
        lp.m = (int32_t)(setV->offsets[id + 1] - setV->offsets[id]);
        lp.nblocks = (int32_t)(((int64_t)lp.m + 1 + kTileRows - 1) / kTileRows);
        lp.ntiles = (lp.n + C - 1) / C;
        lp.p = lp.nblocks * kTileRows - 1 - lp.m;
        const int64_t need = (int64_t)lp.nblocks * (lp.n + 1) * 2 + (int64_t)lp.nblocks * lp.ntiles * kTileRows * 2;
        if (run > 0 && (run + need) * 4 > budget) {
            chunkEnd.push_back(pairs.size());
            run = 0;
        }
        lp.rowck = run;
        lp.colck = run + (int64_t)lp.nblocks * (lp.n + 1) * 2;
        lp.bestck = bestRun;
        bestRun += lp.nblocks;
        run += need;
        maxRun = std::max(maxRun, run);
        pairs.push_back(lp);
    }
    chunkEnd.push_back(pairs.size());
    const size_t np = pairs.size();
    hipError_t err;
    if ((err = ensure(ctx->b.longCk, (size_t)maxRun * 4)) != hipSuccess ||
        (err = ensure(ctx->b.longPairs, sizeof(LongPair) * np)) != hipSuccess ||
        (err = ensure(ctx->b.endEF, (size_t)8 * N)) != hipSuccess ||
        (P.local && (err = ensure(ctx->b.longBest, (size_t)4 * std::max<int64_t>(bestRun, 1))) != hipSuccess))
        return hipFail(ctx, err, "allocating long-pair buffers");
    if (dCounts && ((err = ensure(ctx->b.longWalk, (size_t)4 * kWalkStateInts * np)) != hipSuccess ||
                    (err = ensure(ctx->b.longTrace, sizeof(uint2) * (size_t)kTileRecSteps * 16 * kRoundSlots * np)) !=
                        hipSuccess))
        return hipFail(ctx, err, "allocating long-pair traceback buffers");
    if ((err = hipMemcpyAsync(ctx->b.longPairs.p, pairs.data(), sizeof(LongPair) * np, hipMemcpyHostToDevice,
                              stream)) != hipSuccess)
        return hipFail(ctx, err, "uploading long pairs");
    size_t b = 0;
    for (size_t e : chunkEnd) {
        TileArgs a{};
        a.hRes = in.dH;
        a.vRes = in.dV;
        a.hOff = static_cast<const int64_t *>(ctx->b.hOff.p);
        a.vOff = static_cast<const int64_t *>(ctx->b.vOff.p);
        a.pairs = static_cast<const LongPair *>(ctx->b.longPairs.p) + b;
        a.nPairs = (int32_t)(e - b);
        a.tileC = C;
        a.ck = static_cast<int32_t *>(ctx->b.longCk.p);
        a.gapOpen = P.si.o;
        a.gapExtend = P.si.e;
        a.dnaProfile = static_cast<const uint32_t *>(ctx->b.dnaProf.p);
        a.scores = in.dScores;
        a.endEF = static_cast<int32_t *>(ctx->b.endEF.p);
        a.mode = P.mode;
        a.best = static_cast<int32_t *>(ctx->b.longBest.p);
        a.alpha = P.si.alpha;
        int maxB = 0, maxT = 0;
        for (size_t k = b; k < e; ++k) {
            maxB = std::max(maxB, pairs[k].nblocks);
            maxT = std::max(maxT, pairs[k].ntiles);
        }
        a.wavesPerPair = (maxB + 3) / 4;
        // Every launch sweeps one tile anti-diagonal and ends with a barrier
        // for its whole grid.  Groups of pair couples on separate streams do
        // not wait for each other's slowest tiles, so their launches fill
        // the SIMDs the others leave idle (the ramps of the wavefront and
        // the last waves of the widest anti-diagonals).  Group 0 stays on the
        // call's stream, so that ns groups use ns hardware queues.
        const int couples = (int)((e - b + 1) / 2);
        const int ns = std::min(longStreams(), couples);
        std::vector<TileArgs> sub(ns, a);
        for (int s = 0; s < ns; ++s) {
            const int c0 = couples * s / ns, c1 = couples * (s + 1) / ns;
            sub[s].pairs = a.pairs + 2 * c0;
            sub[s].nPairs = std::min((int32_t)(2 * c1), a.nPairs) - 2 * c0;
        }
        if (ns > 1) {
            if (!ctx->longFork && (err = hipEventCreateWithFlags(&ctx->longFork, hipEventDisableTiming)) != hipSuccess)
                return hipFail(ctx, err, "creating long-pair events");
            for (int s = 1; s < ns; ++s) {
                if (!ctx->longStreams[s] && (err = hipStreamCreate(&ctx->longStreams[s])) != hipSuccess)
                    return hipFail(ctx, err, "creating long-pair streams");
                if (!ctx->longJoin[s] &&
                    (err = hipEventCreateWithFlags(&ctx->longJoin[s], hipEventDisableTiming)) != hipSuccess)
                    return hipFail(ctx, err, "creating long-pair events");
            }
            hipEvent_t fork = ctx->longFork;
            if ((err = op([=] { return hipEventRecord(fork, stream); })) != hipSuccess)
                return hipFail(ctx, err, "long-pair fork");
            for (int s = 1; s < ns; ++s) {
                hipStream_t side = ctx->longStreams[s];
                if ((err = op([=] { return hipStreamWaitEvent(side, fork, 0); })) != hipSuccess)
                    return hipFail(ctx, err, "long-pair fork");
            }
        }
        for (int d = 0; d < maxB + maxT - 1; ++d) {
            for (int s = 0; s < ns; ++s) {
                TileArgs t = sub[s];
                t.diag = d;
                hipStream_t st = s > 0 ? ctx->longStreams[s] : stream;
                if ((err = op([=] { return launchTileFwd32(t, st); })) !=
                    hipSuccess)
                    return hipFail(ctx, err, "launching long-pair forward");
            }
        }
        if (ns > 1) {
            for (int s = 1; s < ns; ++s) {
                hipEvent_t join = ctx->longJoin[s];
                hipStream_t side = ctx->longStreams[s];
                if ((err = op([=] {
                         hipError_t e = hipEventRecord(join, side);
                         return e != hipSuccess ? e : hipStreamWaitEvent(stream, join, 0);
                     })) != hipSuccess)
                    return hipFail(ctx, err, "long-pair join");
            }
        }
        if (P.mode != 0) {
            const TileArgs ta = a;
            if ((err = op([=] { return launchLongResult(ta, stream); })) != hipSuccess)
                return hipFail(ctx, err, "launching long-pair results");
        }
        if (dCounts) {
            a.trace = static_cast<uint2 *>(ctx->b.longTrace.p);
            a.walk = static_cast<int32_t *>(ctx->b.longWalk.p);
            a.counts = dCounts;
            a.ops = rows.ops;
            a.opOff = rows.opOff;
            a.opLen = rows.opLen;
            const TileArgs ta = a;
            if ((err = op([=] { return launchTileWalkInit(ta, stream); })) != hipSuccess)
                return hipFail(ctx, err, "launching long-pair walk init");
            // Each round moves the walk up kRoundBlocks row blocks or left
            // kRoundTiles tiles (or ends it); extra rounds do nothing.
            const int rounds = (maxB + kRoundBlocks - 1) / kRoundBlocks + (maxT + kRoundTiles - 1) / kRoundTiles + 1;
            for (int r = 0; r < rounds; ++r) {
                if ((err = op([=] {
                         hipError_t e = launchTileTrace32(ta, stream);
                         return e != hipSuccess ? e : launchTileWalk32(ta, stream);
                     })) != hipSuccess)
                    return hipFail(ctx, err, "launching long-pair traceback");
            }
        }
        b = e;
    }
    return SQMI_OK;
}

}  // namespace

extern "C" {

int sqmi_abi_version(void) { return SQMI_ABI_VERSION; }

const char *sqmi_status_string(sqmi_status s)
{
    switch (s) {
        case SQMI_OK: return "ok";
        case SQMI_ERR_INVALID_ARGUMENT: return "invalid argument";
        case SQMI_ERR_LENGTH_MISMATCH: return "sequence sets differ in length";
        case SQMI_ERR_UNSUPPORTED: return "unsupported request";
        case SQMI_ERR_NO_DEVICE: return "no usable gfx950 device";
        case SQMI_ERR_DEVICE: return "device error";
        case SQMI_ERR_OUT_OF_MEMORY: return "out of device memory";
    }
    return "unknown status";
}

const char *sqmi_last_error(const sqmi_context *ctx) { return ctx ? ctx->lastError.c_str() : ""; }

sqmi_status sqmi_create(int device, sqmi_context **out)
{
    if (!out)
        return SQMI_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0 || device < 0 || device >= n)
        return SQMI_ERR_NO_DEVICE;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess)
        return SQMI_ERR_NO_DEVICE;
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return SQMI_ERR_NO_DEVICE;
    sqmi_context *ctx = new (std::nothrow) sqmi_context();
    if (!ctx)
        return SQMI_ERR_OUT_OF_MEMORY;
    ctx->planned = new (std::nothrow) Planned();
    if (!ctx->planned) {
        delete ctx;
        return SQMI_ERR_OUT_OF_MEMORY;
    }
    ctx->device = device;
    ctx->numCUs = prop.multiProcessorCount;
    ctx->l2PerCU = (int64_t)prop.l2CacheSize / 32;
    ctx->totalMem = (int64_t)prop.totalGlobalMem;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&ctx->ownStream) != hipSuccess ||
        hipEventCreate(&ctx->ev0) != hipSuccess || hipEventCreate(&ctx->ev1) != hipSuccess ||
        hipHostMalloc(reinterpret_cast<void **>(&ctx->waitFlag), 64, hipHostMallocDefault) != hipSuccess ||
        scratchAddress(device, &ctx->scratchPtr) != hipSuccess) {
        if (ctx->ev0)
            (void)hipEventDestroy(ctx->ev0);
        if (ctx->ev1)
            (void)hipEventDestroy(ctx->ev1);
        if (ctx->ownStream)
            (void)hipStreamDestroy(ctx->ownStream);
        if (ctx->waitFlag)
            (void)hipHostFree(ctx->waitFlag);
        delete ctx->planned;
        delete ctx;
        return SQMI_ERR_DEVICE;
    }
    *ctx->waitFlag = 0;
    ctx->stream = ctx->ownStream;
    *out = ctx;
    return SQMI_OK;
}

sqmi_status sqmi_destroy(sqmi_context *ctx)
{
    if (!ctx)
        return SQMI_OK;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    dropReplay(ctx);
    ctx->b.forEach([](DevBuf &b) { release(b); });
    if (ctx->ev0)
        (void)hipEventDestroy(ctx->ev0);
    if (ctx->ev1)
        (void)hipEventDestroy(ctx->ev1);
    for (int s = 0; s < sqmi_context::kMaxLongStreams; ++s) {
        if (ctx->longJoin[s])
            (void)hipEventDestroy(ctx->longJoin[s]);
        if (ctx->longStreams[s]) {
            (void)hipStreamSynchronize(ctx->longStreams[s]);
            (void)hipStreamDestroy(ctx->longStreams[s]);
        }
    }
    if (ctx->longFork)
        (void)hipEventDestroy(ctx->longFork);
    if (ctx->ownStream)
        (void)hipStreamDestroy(ctx->ownStream);
    release(ctx->stage);
    if (ctx->pin)
        (void)hipHostFree(ctx->pin);
    if (ctx->waitFlag)
        (void)hipHostFree(ctx->waitFlag);
    delete ctx->planned;
    delete ctx;
    return SQMI_OK;
}

sqmi_status sqmi_set_stream(sqmi_context *ctx, void *stream)
{
    if (!ctx)
        return SQMI_ERR_INVALID_ARGUMENT;
    ctx->stream = stream ? reinterpret_cast<hipStream_t>(stream) : ctx->ownStream;
    return SQMI_OK;
}

sqmi_status sqmi_get_stats(const sqmi_context *ctx, sqmi_stats *out)
{
    if (!ctx || !out)
        return SQMI_ERR_INVALID_ARGUMENT;
    *out = ctx->stats;
    return SQMI_OK;
}

}  // extern "C"

// sqmi_align_score and, with ctx->noAlloc, sqmi_align_score_noalloc (every
// ensure() then carves from ctx->arena; the size of the whole request is
// checked before anything is copied or launched, and the row buffers'
// grid is cut to what the arena holds).
static sqmi_status alignScore(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                              const sqmi_scoring *scoring, uint32_t mode, int32_t *scores, uint32_t flags)
{
    const auto tStart = std::chrono::steady_clock::now();
    if (!ctx)
        return SQMI_ERR_INVALID_ARGUMENT;
    ctx->lastError.clear();
    ctx->stats = sqmi_stats{};
    sqmi_status st;
    if ((st = validate(ctx, setH, setV, scoring, mode)) != SQMI_OK || (st = checkForced(ctx, flags)) != SQMI_OK)
        return st;
    const int64_t N = setH->count;
    if (N == 0)
        return SQMI_OK;
    if (!scores)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "scores is null");
    if (hipSetDevice(ctx->device) != hipSuccess)
        return fail(ctx, SQMI_ERR_DEVICE, "hipSetDevice failed");
    hipStream_t stream = ctx->stream;

    // Replay: a call whose plan depends on nothing that differs from the
    // last call's (lengths, scoring, mode, flags, the device addresses the
    // kernels take, the planner's switches) reuses its plan, which is still
    // in the context's device buffers, and relaunches its graph; only host
    // residues and host scores are copied again.
    const bool replayable = graphsEnabled() && !ctx->noAlloc && !(flags & SQMI_PLAIN_PER_PAIR);
    uint64_t key = 0;
    hipError_t err;
    if (replayable) {
        const auto tKey = std::chrono::steady_clock::now();
        key = digest64(setH->offsets, N + 1) ^ mix64(digest64(setV->offsets, N + 1) + 1);
        std::vector<int64_t> scal = {N, mode, flags, scoring->alphabet_size, scoring->gap_open, scoring->gap_extend,
                                     ctx->device};
        for (int k = 0; k < scoring->alphabet_size * scoring->alphabet_size; ++k)
            scal.push_back(scoring->table[k]);
        if (flags & SQMI_RESIDUES_ON_DEVICE) {
            scal.push_back((int64_t)(uintptr_t)setH->residues);
            scal.push_back((int64_t)(uintptr_t)setV->residues);
        }
        if (flags & SQMI_SCORES_ON_DEVICE)
            scal.push_back((int64_t)(uintptr_t)scores);
        scal.push_back((int64_t)(uintptr_t)stream);   // the kept launches name it
        for (const char *name : {"SQMI_COOP_MIN_BLOCKS", "SQMI_LONG_ALL", "SQMI_LONG_MIN_SIDE", "SQMI_LONG_STREAMS", "SQMI_LONG_ROWS",
                                 "SQMI_SHAPE_RULE", "SQMI_TRACE_BUDGET_MB", "SQMI_ROW_UNITS", "SQMI_BIN_SHAPES"}) {
            const char *v = std::getenv(name);
            for (const char *c = v ? v : ""; *c; ++c)
                scal.push_back(*c);
            scal.push_back(-1);
        }
        key ^= mix64(digest64(scal.data(), (int64_t)scal.size()) + 2);
        if (ctx->replay.valid && ctx->replay.key == key) {
            const double keyMs = msSince(tKey);
            const uint8_t *rH = setH->residues, *rV = setV->residues;
            const int64_t hTot = setH->offsets[N], vTot = setV->offsets[N];
            // Residues that were staged are staged again, at their places, and
            // the scores come back through the stage too (by
            // three pageable copies 256 pairs of 150 bp take 122 us, so 82).
            if ((err = stageResume(ctx, downScores(N, flags))) != hipSuccess)
                return hipFail(ctx, err, "waiting for an earlier call");
            if (!(flags & SQMI_RESIDUES_ON_DEVICE)) {
                if (ctx->b.hRes.view && ctx->b.vRes.view)
                    err = restage(ctx, ctx->b.hRes, rH, hTot, ctx->b.vRes, rV, vTot);
                else if ((err = hipMemcpyAsync(ctx->b.hRes.p, rH, hTot, hipMemcpyHostToDevice, stream)) == hipSuccess)
                    err = hipMemcpyAsync(ctx->b.vRes.p, rV, vTot, hipMemcpyHostToDevice, stream);
                if (err != hipSuccess)
                    return hipFail(ctx, err, "copying residues");
            }
            if (!ctx->replay.exec && ctx->replay.launches.size() > kDirectLaunches)
                captureReplay(ctx);
            if ((err = hipEventRecord(ctx->ev0, stream)) != hipSuccess)
                return hipFail(ctx, err, "event");
            if (ctx->replay.exec) {
                if ((err = hipGraphLaunch(ctx->replay.exec, stream)) != hipSuccess)
                    return hipFail(ctx, err, "launching the call's graph");
            } else {
                for (auto &f : ctx->replay.launches)
                    if ((err = f()) != hipSuccess)
                        return hipFail(ctx, err, "launching alignment kernels");
            }
            if ((err = hipEventRecord(ctx->ev1, stream)) != hipSuccess)
                return hipFail(ctx, err, "event");
            if (!(flags & SQMI_SCORES_ON_DEVICE) && (err = fetch(ctx, scores, ctx->b.scores.p, 4 * N)) != hipSuccess)
                return hipFail(ctx, err, "copying scores");
            if ((err = hipStreamSynchronize(stream)) != hipSuccess)
                return hipFail(ctx, err, "alignment kernels");
            deliver(ctx);
            stageEnd(ctx);
            if ((st = stripCheck(ctx)) != SQMI_OK)
                return st;
            ctx->stats = ctx->replay.stats;
            ctx->stats.host_plan_ms = keyMs;
            ctx->stats.replayed = 1;
            float ms = 0;
            ctx->stats.device_ms = hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) == hipSuccess ? ms : 0.0;
            ctx->stats.total_ms = msSince(tStart);
            return SQMI_OK;
        }
    }
    dropReplay(ctx);

    Planned &P = *ctx->planned;
    const PlanUse use{P};
    P.reset();
    const auto tPlan = std::chrono::steady_clock::now();
    plan(*setH, *setV, *scoring, mode, flags, P, false, false,
         ctx->noAlloc ? 0 : std::min(kMaxStripBytes, traceBudget(ctx)));
    if (P.stripWords && ensure(ctx->b.strips, (size_t)P.stripWords * 8) != hipSuccess) {
        // No room for the strips: whole items need a row buffer per wave only.
        (void)hipGetLastError();
        P.reset();
        plan(*setH, *setV, *scoring, mode, flags, P, false, false, 0);
    }
    ctx->stats.host_plan_ms = msSince(tPlan);
    fillStats(P, ctx->stats);
    const ScoringInfo &si = P.si;
    std::vector<Plan16> &plans = P.plans;
    std::vector<int32_t> &emptyIds = P.emptyIds, &ids32 = P.ids32;
    std::vector<int64_t> &scratchOff32 = P.scratchOff32;
    const int64_t scratch32 = P.scratch32;
    const auto &keys16 = P.keys16;
    const uint32_t track = P.track;
    const int kind = P.local ? kScoreLocal : (track & kTrackRight) ? kScoreRight : kScoreGlobal;

    // The no-allocation call: everything but the row buffers has a fixed
    // size; the row buffers need at least one workgroup's worth per shape.
    // A request that does not fit is planned once more in its tightest form.
    size_t rowbufBudget = 0;
    int unitWaves = scoreWaves(P.dna16, (int64_t)P.units.size(), ctx->numCUs);
    RawVec<SlimUnit> slim;
    for (bool tight = false; ctx->noAlloc; tight = true) {
        if (!P.idsLong.empty())
            return fail(ctx, SQMI_ERR_UNSUPPORTED,
                        "sqmi_align_score_noalloc: pairs on the long-pair route need sqmi_align_score");
        const int64_t A2 = (int64_t)si.alpha * si.alpha, hTot = setH->offsets[N], vTot = setV->offsets[N];
        const size_t nSlim = (P.units.size() + 3) / 4 * 4;   // the lists after them start on 16 bytes
        size_t need = 0;
        if (!(flags & SQMI_RESIDUES_ON_DEVICE))
            need += arenaBytes(hTot + 64) + arenaBytes(vTot + 64);
        need += 2 * arenaBytes(8 * (N + 1));
        if (!(flags & SQMI_SCORES_ON_DEVICE))
            need += arenaBytes(4 * N);
        need += arenaBytes(2 * (si.alpha + 1) * (si.alpha + 1)) + arenaBytes(64) + arenaBytes(4 * A2);
        size_t nOrder = 0, nItems = 0, laneRb = 0;
        for (const Plan16 &pl : plans) {
            nOrder += pl.order.size();
            nItems += pl.items.size();
            laneRb = std::max(laneRb, (size_t)wavesPerBlock16() * 64 * laneRowCols(pl.maxN, pl.var.R) * 8);
        }
        if (!plans.empty())
            need += arenaBytes(4 * nOrder) + arenaBytes(sizeof(WorkItem) * nItems);
        if (!P.units.empty())
            need += arenaBytes(4 * P.order16.size()) + arenaBytes(sizeof(SlimUnit) * nSlim);
        if (!plans.empty() || !P.units.empty())
            need += arenaBytes(64 * (plans.size() + 1));
        if (!ids32.empty())
            need += arenaBytes(4 * ids32.size()) + arenaBytes(8 * ids32.size()) + arenaBytes((size_t)8 * scratch32);
        if (!emptyIds.empty())
            need += arenaBytes(4 * emptyIds.size());
        const size_t cap = ctx->arena.cap - ctx->arena.used;
        unitWaves = scoreWaves(P.dna16, (int64_t)P.units.size(), ctx->numCUs);
        auto rowbufs = [&] { return arenaBytes(std::max(laneRb, (size_t)unitWaves * P.slotWords * 8)); };
        if (need + rowbufs() > cap)
            unitWaves = std::min(unitWaves, 4);
        if (need + rowbufs() <= cap) {
            rowbufBudget = (cap - need) & ~(size_t)255;   // holds rowbufs()
            slim.resize(nSlim);
            for (size_t k = 0; k < nSlim; ++k)
                slim[k] = k < P.units.size() ? SlimUnit::of(P.units[k]) : SlimUnit{};
            break;
        }
        if (tight)
            return fail(ctx, SQMI_ERR_OUT_OF_MEMORY,
                        "sqmi_align_score_noalloc: the request needs " + std::to_string(need + rowbufs()) +
                            " bytes of device scratch, more than the " + std::to_string(cap) +
                            " of SQMI_NOALLOC_SCRATCH_BYTES; use sqmi_align_score");
        P.reset();
        plan(*setH, *setV, *scoring, mode, flags, P, false, false, 0, true);
        fillStats(P, ctx->stats);
    }

    // ---- device buffers --------------------------------------------------
    Inputs in;
    {
        // Offsets, tables and the packed kernels' lists; the other routes'
        // lists are copied by themselves.
        size_t bytes = stageInputs(setH, setV, scoring, flags) + stageBytes(4 * (P.order16.size() + (size_t)N)) +
                       stageBytes(sizeof(ScoreUnit) * P.units.size());
        for (const Plan16 &pl : plans)
            bytes += stageBytes(sizeof(WorkItem) * pl.items.size()) + 256;
        if ((err = stageBegin(ctx, bytes + 1024, downScores(N, flags))) != hipSuccess)
            return hipFail(ctx, err, "allocating upload staging");
    }
    if ((st = uploadInputs(ctx, setH, setV, scoring, si, scores, flags, in)) != SQMI_OK)
        return st;
    const uint8_t *dH = in.dH, *dV = in.dV;
    int32_t *dScores = in.dScores;
    const int A = si.alpha;
    // Kernel launches wait in `launches` until every upload is enqueued.
    Deferred launches;

    // ---- packed score kernel: its arguments but for the units ----------
    ScoreArgs sa{};
    sa.hRes = dH;
    sa.vRes = dV;
    sa.hOff = static_cast<const int64_t *>(ctx->b.hOff.p);
    sa.vOff = static_cast<const int64_t *>(ctx->b.vOff.p);
    sa.error = ctx->waitFlag;
    sa.scores = dScores;
    sa.mode = mode;
    sa.alpha = A;
    sa.tTable = static_cast<const int16_t *>(ctx->b.tTable.p);
    sa.dnaProfile = static_cast<const uint32_t *>(ctx->b.dnaProf.p);
    sa.drift = P.drift;

    // ---- plain form: one launch per pair (baseline for the batched form) --
    // Host data staged by hipMemcpyAsync must outlive the copies: the plain
    // form's lists live at function scope, like the planner's.
    std::vector<int32_t> plainIds;
    std::vector<ScoreUnit> plainUnits;
    if (flags & SQMI_PLAIN_PER_PAIR) {
        // Its kernels are launched right here: they need the offsets and tables.
        if ((err = stageFlush(ctx)) != hipSuccess)
            return hipFail(ctx, err, "uploading");
        if ((err = hipEventRecord(ctx->ev0, stream)) != hipSuccess)
            return hipFail(ctx, err, "event");
        // One wavefront, whose first 16-lane group sweeps the pair (the other
        // pair slots of the wavefront stay empty).
        int64_t slotWords = 1;
        for (const Key &k : keys16) {
            const int32_t id = k.id;
            const int64_t n = setH->offsets[id + 1] - setH->offsets[id];
            const int64_t m = setV->offsets[id + 1] - setV->offsets[id];
            const int units = (int)unitsOfRows(m), nb = (units + 3) / 4;
            plainUnits.push_back(ScoreUnit{(int32_t)plainIds.size(), 1, (int32_t)n, nb,
                                           16 | (4 * (units - 4 * (nb - 1))) << 8,
                                           driftNarrow(si, P.drift, P.local, n, m) ? 0 : kUnitWide, -1, 0, 0});
            plainIds.push_back(id);
            slotWords = std::max<int64_t>(slotWords, 4 * (n + 1));
        }
        const size_t np = plainIds.size();
        if ((err = ensure(ctx->b.order, 4 * np)) != hipSuccess ||
            (err = ensure(ctx->b.items, sizeof(ScoreUnit) * np)) != hipSuccess ||
            (err = ensure(ctx->b.queue, 4 * np + 64)) != hipSuccess ||
            (err = ensure(ctx->b.rowbuf, (size_t)slotWords * 8)) != hipSuccess)
            return hipFail(ctx, err, "allocating plain work lists");
        if (np && ((err = hipMemcpyAsync(ctx->b.order.p, plainIds.data(), 4 * np, hipMemcpyHostToDevice, stream)) !=
                       hipSuccess ||
                   (err = hipMemcpyAsync(ctx->b.items.p, plainUnits.data(), sizeof(ScoreUnit) * np,
                                         hipMemcpyHostToDevice, stream)) != hipSuccess ||
                   (err = hipMemsetAsync(ctx->b.queue.p, 0, 4 * np, stream)) != hipSuccess))
            return hipFail(ctx, err, "uploading plain work lists");
        for (size_t k = 0; k < np; ++k) {
            ScoreArgs a = sa;
            a.order = static_cast<const int32_t *>(ctx->b.order.p);
            a.units = static_cast<const ScoreUnit *>(ctx->b.items.p) + k;
            a.nUnits = 1;
            a.queue = static_cast<uint32_t *>(ctx->b.queue.p) + k;
            a.rowbuf = static_cast<uint64_t *>(ctx->b.rowbuf.p);
            a.slotWords = slotWords;
            if ((err = launchScore16(P.dna16, kind, a, 1, 1, stream)) != hipSuccess)
                return hipFail(ctx, err, "launching plain kernel");
        }
        plans.clear();
        P.units.clear();
    }

    // ---- packed int16 kernels -------------------------------------------
    // The packed score kernel takes every group unit in one launch; the
    // one-pair-per-lane shapes in use one launch each, in order on the
    // stream.  Each has its own slices of the work lists and its own queue
    // counter (cleared by one fill kernel), so the uploads of a later launch
    // never touch what an earlier one still reads; the launches share the row
    // buffers, which a launch only uses while it runs.
    if (!plans.empty() || !P.units.empty()) {
        const int wpb = wavesPerBlock16();
        const size_t unitBytes = ctx->noAlloc ? sizeof(SlimUnit) * slim.size() : sizeof(ScoreUnit) * P.units.size();
        const size_t unitOrder = P.order16.size();
        std::vector<size_t> orderOff(plans.size() + 1, unitOrder), itemOff(plans.size() + 1, 0);
        std::vector<int> grids(plans.size()), rowColsOf(plans.size());
        size_t rbMax = 0;
        int unitGrid = 0;
        if (!P.units.empty()) {
            unitGrid = std::max(1, (int)std::min<int64_t>((int64_t)ctx->numCUs * occupancyScore16(P.dna16, kind, unitWaves),
                                                          ((int64_t)P.units.size() + unitWaves - 1) / unitWaves));
            const size_t perBlock = std::max<size_t>((size_t)unitWaves * P.slotWords * 8, 8);
            if (ctx->noAlloc)   // the persistent grid shrinks to the scratch that is left
                unitGrid = (int)std::max<size_t>(1, std::min<size_t>((size_t)unitGrid, rowbufBudget / perBlock));
            rbMax = (size_t)unitGrid * perBlock;
        }
        for (size_t k = 0; k < plans.size(); ++k) {
            const Plan16 &pl = plans[k];
            const Variant16 &v = pl.var;
            if (!laneSupported(v))
                return fail(ctx, SQMI_ERR_UNSUPPORTED, "kernel variant not compiled");
            const int64_t nIt = (int64_t)pl.items.size();
            grids[k] = std::max(1, (int)std::min<int64_t>((int64_t)ctx->numCUs * occupancyLane16(v), (nIt + wpb - 1) / wpb));
            // Row buffers per wave slot: one per lane, column-major across the 64 lanes.
            rowColsOf[k] = laneRowCols(pl.maxN, v.R);
            const size_t perBlock = (size_t)wpb * 64 * rowColsOf[k] * 8;
            if (ctx->noAlloc)
                grids[k] = (int)std::max<size_t>(1, std::min<size_t>((size_t)grids[k], rowbufBudget / perBlock));
            rbMax = std::max(rbMax, (size_t)grids[k] * perBlock);
            orderOff[k + 1] = orderOff[k] + pl.order.size();
            itemOff[k + 1] = itemOff[k] + pl.items.size();
        }
        const size_t nq = 16 * (plans.size() + 1);   // queue counters: 16 dwords per launch
        std::vector<Piece> orders, lists;
        if (!P.units.empty()) {
            orders.push_back({P.order16.data(), 4 * unitOrder});
            lists.push_back({ctx->noAlloc ? (const void *)slim.data() : P.units.data(), unitBytes});
        }
        for (const Plan16 &pl : plans) {
            orders.push_back({pl.order.data(), 4 * pl.order.size()});
            lists.push_back({pl.items.data(), sizeof(WorkItem) * pl.items.size()});
        }
        if ((err = put(ctx, ctx->b.order, orders.data(), orders.size())) != hipSuccess ||
            (err = put(ctx, ctx->b.items, lists.data(), lists.size())) != hipSuccess)
            return hipFail(ctx, err, "uploading work lists");
        if ((err = ensure(ctx->b.queue, 4 * nq)) != hipSuccess || (err = ensure(ctx->b.rowbuf, rbMax)) != hipSuccess)
            return hipFail(ctx, err, "allocating work lists");
        uint32_t *dQueues = static_cast<uint32_t *>(ctx->b.queue.p);
        launches.push_back([=] { return launchZero32(dQueues, nq, stream); });
        if (!P.units.empty()) {
            ScoreArgs a = sa;
            a.order = static_cast<const int32_t *>(ctx->b.order.p);
            a.units = static_cast<const ScoreUnit *>(ctx->b.items.p);
            a.slim = ctx->noAlloc ? static_cast<const SlimUnit *>(ctx->b.items.p) : nullptr;
            a.nUnits = (int32_t)P.units.size();
            a.queue = dQueues;
            a.rowbuf = static_cast<uint64_t *>(ctx->b.rowbuf.p);
            a.slotWords = P.slotWords;
            a.strips = static_cast<uint64_t *>(ctx->b.strips.p);
            a.stripWords = P.stripWords;
            if (P.stripWords > 0) {
                // Strips find their input words by their not being 0, and
                // merge the results of modes that track every block's cells.
                const size_t words = 2 * (size_t)P.stripWords;
                uint32_t *dStrips = static_cast<uint32_t *>(ctx->b.strips.p);
                launches.push_back([=] { return launchZero32(dStrips, words, stream); });
                if (kind != kScoreGlobal)
                    launches.push_back([=] {
                        return launchFill32(reinterpret_cast<uint32_t *>(dScores), (size_t)N, (uint32_t)INT32_MIN, stream);
                    });
            }
            const bool dna = P.dna16;
            launches.push_back([=] { return launchScore16(dna, kind, a, unitGrid, unitWaves, stream); });
        }
        for (size_t k = 0; k < plans.size(); ++k) {
            const Plan16 &pl = plans[k];
            const Variant16 &v = pl.var;
            int32_t *dOrder = static_cast<int32_t *>(ctx->b.order.p) + orderOff[k];
            WorkItem *dItems = reinterpret_cast<WorkItem *>(static_cast<char *>(ctx->b.items.p) + unitBytes) + itemOff[k];
            FwdArgs a{};
            a.hRes = dH;
            a.vRes = dV;
            a.hOff = static_cast<const int64_t *>(ctx->b.hOff.p);
            a.vOff = static_cast<const int64_t *>(ctx->b.vOff.p);
            a.order = dOrder;
            a.items = dItems;
            a.nItems = (int32_t)pl.items.size();
            a.queue = dQueues + 16 * (k + 1);
            a.rowbuf = static_cast<uint32_t *>(ctx->b.rowbuf.p);
            a.rowCols = rowColsOf[k];
            a.scores = dScores;
            a.gapOpen = si.o;
            a.gapExtend = si.e;
            a.mode = mode;
            a.alpha = A;
            a.tTable = static_cast<const int16_t *>(ctx->b.tTable.p);
            a.dnaProfile = static_cast<const uint32_t *>(ctx->b.dnaProf.p);
            a.drift = P.drift;
            const int grid = grids[k];
            launches.push_back([=] { return launchLane16(v, a, grid, stream); });
        }
    }

    // ---- int32 pairs -------------------------------------------------------
    if (!ids32.empty()) {
        const size_t n32 = ids32.size();
        if ((err = ensure(ctx->b.ids32, 4 * n32)) != hipSuccess ||
            (err = ensure(ctx->b.scratchOff32, 8 * n32)) != hipSuccess ||
            (err = ensure(ctx->b.scratch32, (size_t)8 * scratch32)) != hipSuccess)
            return hipFail(ctx, err, "allocating int32 lists");
        if ((err = hipMemcpyAsync(ctx->b.ids32.p, ids32.data(), 4 * n32, hipMemcpyHostToDevice, stream)) != hipSuccess ||
            (err = hipMemcpyAsync(ctx->b.scratchOff32.p, scratchOff32.data(), 8 * n32, hipMemcpyHostToDevice, stream)) !=
                hipSuccess)
            return hipFail(ctx, err, "uploading int32 lists");
        Simple32Args a{};
        a.hRes = dH;
        a.vRes = dV;
        a.hOff = static_cast<const int64_t *>(ctx->b.hOff.p);
        a.vOff = static_cast<const int64_t *>(ctx->b.vOff.p);
        a.ids = static_cast<const int32_t *>(ctx->b.ids32.p);
        a.scratchOff = static_cast<const int64_t *>(ctx->b.scratchOff32.p);
        a.nIds = (int32_t)n32;
        a.scratch = static_cast<int32_t *>(ctx->b.scratch32.p);
        a.scores = dScores;
        a.gapOpen = si.o;
        a.gapExtend = si.e;
        a.mode = mode;
        a.alpha = A;
        a.table = static_cast<const int32_t *>(ctx->b.table32.p);
        launches.push_back([=] { return launchSimple32(a, stream); });
    }
    LongStage longStage;
    if ((st = runLong(ctx, setH, setV, P, in, flags, nullptr, RowsDev{}, longStage, &launches)) != SQMI_OK)
        return st;
    if (!emptyIds.empty()) {
        if ((err = ensure(ctx->b.emptyIds, 4 * emptyIds.size())) != hipSuccess)
            return hipFail(ctx, err, "allocating empty list");
        if ((err = hipMemcpyAsync(ctx->b.emptyIds.p, emptyIds.data(), 4 * emptyIds.size(), hipMemcpyHostToDevice,
                                  stream)) != hipSuccess)
            return hipFail(ctx, err, "uploading empty list");
        const int ne = (int)emptyIds.size();
        const int32_t *dEmpty = static_cast<const int32_t *>(ctx->b.emptyIds.p);
        launches.push_back([=] { return launchFillScores(dScores, dEmpty, ne, INT32_MIN, stream); });
    }

    // ---- the launches: run, and kept for an identical next call ----------
    if ((err = stageFlush(ctx)) != hipSuccess)
        return hipFail(ctx, err, "uploading");
    if (!(flags & SQMI_PLAIN_PER_PAIR) && (err = hipEventRecord(ctx->ev0, stream)) != hipSuccess)
        return hipFail(ctx, err, "event");
    for (auto &f : launches)
        if ((err = f()) != hipSuccess)
            return hipFail(ctx, err, "launching alignment kernels");
    if ((err = hipEventRecord(ctx->ev1, stream)) != hipSuccess)
        return hipFail(ctx, err, "event");
    if (!(flags & SQMI_SCORES_ON_DEVICE)) {
        if ((err = fetch(ctx, scores, dScores, 4 * N)) != hipSuccess)
            return hipFail(ctx, err, "copying scores");
    }
    if ((err = hipStreamSynchronize(stream)) != hipSuccess)
        return hipFail(ctx, err, "alignment kernels");
    deliver(ctx);
    stageEnd(ctx);
    if ((st = stripCheck(ctx)) != SQMI_OK)
        return st;
    float ms = 0;
    if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) == hipSuccess)
        ctx->stats.device_ms = ms;
    ctx->stats.total_ms = msSince(tStart);
    if (replayable && !launches.empty()) {
        ctx->replay.valid = true;
        ctx->replay.key = key;
        ctx->replay.launches = std::move(launches);
        ctx->replay.stats = ctx->stats;
    }
    return SQMI_OK;
}

extern "C" {

sqmi_status sqmi_align_score(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                             const sqmi_scoring *scoring, uint32_t mode, int32_t *scores, uint32_t flags)
{
    return alignScore(ctx, setH, setV, scoring, mode, scores, flags);
}

// The context's buffers are set aside for the call and replaced by empty ones
// that carve from the device's scratch array (ctx->scratchPtr, looked up at
// sqmi_create); afterwards the arena pieces are dropped (nothing to free)
// and the context's own buffers come back untouched.
sqmi_status sqmi_align_score_noalloc(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                                     const sqmi_scoring *scoring, uint32_t mode, int32_t *scores, uint32_t flags)
{
    if (!ctx)
        return SQMI_ERR_INVALID_ARGUMENT;
    if (flags & SQMI_PLAIN_PER_PAIR)
        return fail(ctx, SQMI_ERR_UNSUPPORTED, "sqmi_align_score_noalloc: no plain form");
    if (!ctx->scratchPtr)
        return fail(ctx, SQMI_ERR_DEVICE, "sqmi_align_score_noalloc: no device scratch on this context");
    dropReplay(ctx);
    Buffers own;
    std::swap(own, ctx->b);
    ctx->arena = Arena{static_cast<char *>(ctx->scratchPtr), kNoAllocScratchBytes, 0};
    ctx->b.forEach([&](DevBuf &d) { d.arena = &ctx->arena; });
    ctx->noAlloc = true;
    const sqmi_status st = alignScore(ctx, setH, setV, scoring, mode, scores, flags);
    ctx->noAlloc = false;
    std::swap(own, ctx->b);
    ctx->arena = Arena{};
    return st;
}

sqmi_status sqmi_plan_stats(const sqmi_sequences *setH, const sqmi_sequences *setV, const sqmi_scoring *scoring,
                            uint32_t mode, uint32_t flags, sqmi_stats *out)
{
    if (!out)
        return SQMI_ERR_INVALID_ARGUMENT;
    *out = sqmi_stats{};
    sqmi_status st;
    if ((st = validate(nullptr, setH, setV, scoring, mode)) != SQMI_OK || (st = checkForced(nullptr, flags)) != SQMI_OK)
        return st;
    Planned P;
    const auto t0 = std::chrono::steady_clock::now();
    plan(*setH, *setV, *scoring, mode, flags, P);
    out->host_plan_ms = msSince(t0);
    fillStats(P, *out);
    return SQMI_OK;
}

// Traceback: the packed forward pass writes 4 trace bits per cell into a
// buffer of at most traceBudget() bytes, so the work items run in chunks;
// after each chunk 16 or 64 lanes per pair walk its path.  Banded pairs (band
// given) whose band has at most kMaxBandTrace diagonals inside the matrix run
// the banded trace kernels (one byte per cell of the band); wider bands, pairs
// outside the int16 window and every pair under SQMI_FORCE_INT32 run the int32
// kernel with one trace byte per cell of the matrix.  All are chunked by the
// same budget.
static sqmi_status alignBackward(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                                 const sqmi_scoring *scoring, uint32_t mode, int32_t *scores, int32_t *counts,
                                 uint8_t *ops, const int64_t *opOffsets, int64_t *opLengths, int64_t *begins,
                                 uint32_t flags, const int64_t *band = nullptr)
{
    const auto tStart = std::chrono::steady_clock::now();
    const bool wantRows = ops != nullptr;
    if (!ctx)
        return SQMI_ERR_INVALID_ARGUMENT;
    dropReplay(ctx);   // this call rewrites the buffers a replay would reuse
    ctx->lastError.clear();
    ctx->stats = sqmi_stats{};
    sqmi_status st;
    if ((st = validate(ctx, setH, setV, scoring, mode)) != SQMI_OK)
        return st;
    if (flags & (SQMI_PLAIN_PER_PAIR | 0x00FFFF00u))
        return fail(ctx, SQMI_ERR_UNSUPPORTED, "sqmi_align_counts: no plain form or forced shapes");
    const int64_t N = setH->count;
    if (N == 0)
        return SQMI_OK;
    if (!scores || !counts)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "scores or counts is null");
    if (wantRows) {
        if (!opOffsets || !opLengths)
            return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "op_offsets or op_lengths is null");
        if (opOffsets[0] < 0)
            return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "op_offsets[0] is negative");
        for (int64_t i = 0; i < N; ++i) {
            const int64_t need = (setH->offsets[i + 1] - setH->offsets[i]) + (setV->offsets[i + 1] - setV->offsets[i]);
            if (opOffsets[i + 1] - opOffsets[i] < need)
                return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "op segment " + std::to_string(i) + " holds fewer than |H| + |V| bytes");
        }
    }
    if (hipSetDevice(ctx->device) != hipSuccess)
        return fail(ctx, SQMI_ERR_DEVICE, "hipSetDevice failed");
    hipStream_t stream = ctx->stream;

    Planned &P = *ctx->planned;
    const PlanUse use{P};
    P.reset();
    Inputs in;
    // Host residue sets of 4 MB and more are copied in on a second host
    // thread while this one plans (the planner reads only the offsets; a
    // pageable copy holds its thread until the data is staged).  On 65,536
    // banded pairs of 150 bp: 3.9-4.2 ms per rows call against 4.4-4.7.
    hipError_t upErr = hipSuccess;
    JoinedThread up;
    if (!(flags & SQMI_RESIDUES_ON_DEVICE) && setH->offsets[N] + setV->offsets[N] >= ((int64_t)4 << 20))
        up.t = std::thread([&] {
            upErr = hipSetDevice(ctx->device);
            if (upErr == hipSuccess)
                upErr = uploadResidues(ctx, setH, setV, in);
        });
    const auto tPlan = std::chrono::steady_clock::now();
    // Banded pairs run on the int32 kernel, band-masked.
    plan(*setH, *setV, *scoring, mode, band ? (flags | SQMI_FORCE_INT32) : flags, P, true, band != nullptr);
    ctx->stats.host_plan_ms = msSince(tPlan);
    up.join();
    if (upErr != hipSuccess)
        return hipFail(ctx, upErr, "copying residues");
    fillStats(P, ctx->stats);
    const ScoringInfo &si = P.si;
    const int A = si.alpha, S = A * A + 2;
    const int64_t budget = traceBudget(ctx);

    // Host-side chunking of the int16 items and of the int32 pairs.  An
    // item's blocks become strips when a wave would take more than a quarter
    // of the chunk's time for it (3,072 resident waves), as in the score
    // calls; SQMI_COOP_MIN_BLOCKS as there.
    const Plan16 *pl = P.plans.empty() ? nullptr : &P.plans[0];
    std::vector<int64_t> itemOff, endOff;   // per item: first record within its chunk (steps), first end candidate
    std::vector<size_t> chunkEnd, chunkUnits;   // item and unit index after each chunk
    RawVec<TraceLoc> locs;                  // per pair in plan order
    int64_t traceRecs = 0;                  // largest chunk, in steps
    int64_t slotWords = 1, stripWords = 0, nEnds = 0;
    std::vector<int64_t> chunkStrips;       // strip words of each chunk
    std::vector<TraceItem> tItems;
    if (pl) {
        traceItems(*setH, *pl, P.dna16, tItems);
        const size_t nIt = tItems.size();
        const int64_t recBytes = 64 * 16;
        itemOff.resize(nIt);
        endOff.resize(nIt);
        locs.resize(pl->order.size());
        std::vector<uint8_t> wide(nIt);
        int64_t run = 0;
        for (size_t k = 0; k < nIt; ++k) {
            const TraceItem &w = tItems[k];
            const int64_t recs = traceRecsOf(w);
            if (run > 0 && (run + recs) * recBytes > budget) {
                chunkEnd.push_back(k);
                run = 0;
            }
            itemOff[k] = run;
            run += recs;
            traceRecs = std::max(traceRecs, run);
        }
        chunkEnd.push_back(nIt);
#pragma omp parallel for schedule(static) if (N > kParallelMin)
        for (int64_t k = 0; k < (int64_t)nIt; ++k) {
            const TraceItem &w = tItems[k];
            bool any = false;
            for (int x = 0; x < w.count; ++x) {
                const int32_t pid = pl->order[w.first + x];
                any |= !driftNarrow(si, P.drift, P.local, setH->offsets[pid + 1] - setH->offsets[pid],
                                    setV->offsets[pid + 1] - setV->offsets[pid]);
            }
            wide[k] = any;
        }
        const int minBlocks = stripMinBlocks();
        P.units.clear();
        for (size_t c = 0, b = 0; c < chunkEnd.size(); b = chunkEnd[c], ++c) {
            int64_t total = 0, off = 0;
            for (size_t k = b; k < chunkEnd[c]; ++k)
                total += (int64_t)tItems[k].nblocks * traceSteps(tItems[k].maxN, tItems[k].lanes);
            for (size_t k = b; k < chunkEnd[c]; ++k) {
                const TraceItem &w = tItems[k];
                const int64_t steps = traceSteps(w.maxN, w.lanes), words = (int64_t)(64 / w.lanes) * (w.maxN + 1);
                const bool strips = w.nblocks > 1 &&
                                    (minBlocks < 0 ? w.lanes == 64 || w.nblocks * steps * 4 * kResidentWaves > total
                                                   : minBlocks > 0 && w.nblocks >= minBlocks);
                const int R = kTraceRows / w.lanes;
                ScoreUnit u{w.first, w.count, w.maxN, w.nblocks, R | R << 8,
                            (wide[k] ? kUnitWide : 0) | (w.lanes == 64 ? kUnit64 : 0), -1, (int32_t)(k - b), 0};
                endOff[k] = nEnds;
                nEnds += (int64_t)w.count * (strips ? w.nblocks : 1);
                if (strips) {
                    u.rowOff = off;
                    off += words * w.nblocks;
                    for (u.block = 0; u.block < w.nblocks; ++u.block)
                        P.units.push_back(u);
                } else {
                    slotWords = std::max<int64_t>(slotWords, words);
                    P.units.push_back(u);
                }
                wide[k] = strips;   // from here on: whether the item has strips
            }
            orderStrips(P.units, chunkUnits.empty() ? 0 : chunkUnits.back());
            chunkUnits.push_back(P.units.size());
            chunkStrips.push_back(off);
            stripWords = std::max(stripWords, off);
        }
#pragma omp parallel for schedule(static) if (N > kParallelMin)
        for (int64_t k = 0; k < (int64_t)nIt; ++k) {
            const TraceItem &w = tItems[k];
            for (int x = 0; x < w.count; ++x) {
                const int32_t pid = pl->order[w.first + x];
                const int64_t m = setV->offsets[pid + 1] - setV->offsets[pid];
                locs[w.first + x] = TraceLoc{itemOff[k], traceSteps(w.maxN, w.lanes),
                                             (int32_t)((int64_t)w.nblocks * kTraceRows - 1 - m), (x / 2) * kTraceLanes, x % 2,
                                             w.lanes, endOff[k] + x, w.count, wide[k] ? w.nblocks : 1, 0};
            }
        }
    }
    std::vector<size_t> chunk32End;         // int32 pairs per chunk
    std::vector<int64_t> off32(P.ids32.size());
    int64_t scratch32 = 0;
    {
        int64_t run = 0;
        for (size_t k = 0; k < P.ids32.size(); ++k) {
            const int64_t need = (k + 1 < P.ids32.size() ? P.scratchOff32[k + 1] : P.scratch32) - P.scratchOff32[k];
            if (need > std::max<int64_t>(budget, (int64_t)4 << 30))
                return fail(ctx, SQMI_ERR_UNSUPPORTED, "sqmi_align_counts: pair too large for the int32 traceback");
            if (run > 0 && run + need > budget) {
                chunk32End.push_back(k);
                run = 0;
            }
            off32[k] = run;
            run += need;
            scratch32 = std::max(scratch32, run);
        }
        if (!P.ids32.empty())
            chunk32End.push_back(P.ids32.size());
    }

    // ---- device buffers --------------------------------------------------
    hipError_t err;
    {
        size_t bytes = stageInputs(setH, setV, scoring, flags) + stageBytes(8 * (N + 1)) + stageBytes(4 * P.ids32.size()) + stageBytes(8 * P.ids32.size()) + 4096;
        if (pl)
            bytes += stageBytes(4 * pl->order.size()) + stageBytes(sizeof(ScoreUnit) * P.units.size()) +
                     2 * stageBytes(8 * tItems.size()) + stageBytes(sizeof(TraceLoc) * pl->order.size());
        size_t down = downScores(N, flags);
        if (down) {
            down += stageBytes((size_t)4 * S * N) + 256;
            if (wantRows)
                down += stageBytes(8 * N) + stageBytes(16 * N) + stageBytes((size_t)(opOffsets[N] - opOffsets[0]));
        }
        if ((err = stageBegin(ctx, bytes, down)) != hipSuccess)
            return hipFail(ctx, err, "allocating upload staging");
    }
    if ((st = uploadInputs(ctx, setH, setV, scoring, si, scores, flags, in)) != SQMI_OK)
        return st;
    int32_t *dCounts = counts;
    if (!(flags & SQMI_SCORES_ON_DEVICE)) {
        if ((err = ensure(ctx->b.counts, (size_t)4 * S * N)) != hipSuccess)
            return hipFail(ctx, err, "allocating counts");
        dCounts = static_cast<int32_t *>(ctx->b.counts.p);
    }
    if ((err = hipMemsetAsync(dCounts, 0, (size_t)4 * S * N, stream)) != hipSuccess)
        return hipFail(ctx, err, "clearing counts");
    RowsDev rows;
    if (wantRows) {
        // Offsets always come from the host; ops and lengths live where the
        // scores do.
        const int64_t opBytes = opOffsets[N];
        if ((err = put(ctx, ctx->b.opOff, opOffsets, 8 * (N + 1))) != hipSuccess)
            return hipFail(ctx, err, "uploading op offsets");
        rows.opOff = static_cast<const int64_t *>(ctx->b.opOff.p);
        if (flags & SQMI_SCORES_ON_DEVICE) {
            rows.ops = ops;
            rows.opLen = opLengths;
        } else {
            if ((err = ensure(ctx->b.ops, (size_t)std::max<int64_t>(opBytes, 1))) != hipSuccess ||
                (err = ensure(ctx->b.opLen, 8 * N)) != hipSuccess)
                return hipFail(ctx, err, "allocating rows");
            rows.ops = static_cast<uint8_t *>(ctx->b.ops.p);
            rows.opLen = static_cast<int64_t *>(ctx->b.opLen.p);
        }
        if ((err = hipMemsetAsync(rows.opLen, 0, 8 * N, stream)) != hipSuccess)
            return hipFail(ctx, err, "clearing op lengths");
        if (begins) {
            if (flags & SQMI_SCORES_ON_DEVICE) {
                rows.begins = begins;
            } else {
                if ((err = ensure(ctx->b.begins, 16 * N)) != hipSuccess)
                    return hipFail(ctx, err, "allocating begins");
                rows.begins = static_cast<int64_t *>(ctx->b.begins.p);
            }
            if ((err = hipMemsetAsync(rows.begins, 0, 16 * N, stream)) != hipSuccess)
                return hipFail(ctx, err, "clearing begins");
        }
    }
    if ((err = hipEventRecord(ctx->ev0, stream)) != hipSuccess)
        return hipFail(ctx, err, "event");

    if (pl) {
        const size_t nIt = tItems.size(), np = pl->order.size();
        const int wpb = wavesPerBlock16();
        size_t maxUnits = 0;
        for (size_t c = 0, b = 0; c < chunkUnits.size(); b = chunkUnits[c], ++c)
            maxUnits = std::max(maxUnits, chunkUnits[c] - b);
        const int grid = std::max(1, (int)std::min<int64_t>((int64_t)ctx->numCUs * occupancyTrace16(P.dna16, P.track),
                                                            ((int64_t)maxUnits + wpb - 1) / wpb));
        if ((err = ensure(ctx->b.queue, 4 * chunkEnd.size() + 64)) != hipSuccess ||
            (err = ensure(ctx->b.rowbuf, (size_t)grid * wpb * slotWords * 8)) != hipSuccess ||
            (err = ensure(ctx->b.strips, (size_t)stripWords * 8)) != hipSuccess ||
            (err = ensure(ctx->b.ends, sizeof(TraceEnd) * (size_t)nEnds)) != hipSuccess ||
            (err = ensure(ctx->b.trace, (size_t)traceRecs * 64 * 16)) != hipSuccess)
            return hipFail(ctx, err, "allocating traceback buffers");
        if ((err = put(ctx, ctx->b.order, pl->order.data(), 4 * np)) != hipSuccess ||
            (err = put(ctx, ctx->b.items, P.units.data(), sizeof(ScoreUnit) * P.units.size())) != hipSuccess ||
            (err = put(ctx, ctx->b.traceOff, itemOff.data(), 8 * nIt)) != hipSuccess ||
            (err = put(ctx, ctx->b.endOff, endOff.data(), 8 * nIt)) != hipSuccess ||
            (err = put(ctx, ctx->b.locs, locs.data(), sizeof(TraceLoc) * np)) != hipSuccess ||
            (err = stageFlush(ctx)) != hipSuccess ||
            (err = hipMemsetAsync(ctx->b.queue.p, 0, 4 * chunkEnd.size() + 64, stream)) != hipSuccess)
            return hipFail(ctx, err, "uploading traceback work lists");
        const int32_t *dOrder = static_cast<const int32_t *>(ctx->b.order.p);
        size_t b = 0, ub = 0;
        for (size_t c = 0; c < chunkEnd.size(); ++c) {
            const size_t e = chunkEnd[c], ue = chunkUnits[c];
            TraceArgs a{};
            a.hRes = in.dH;
            a.vRes = in.dV;
            a.hOff = static_cast<const int64_t *>(ctx->b.hOff.p);
            a.vOff = static_cast<const int64_t *>(ctx->b.vOff.p);
            a.order = dOrder;
            a.units = static_cast<const ScoreUnit *>(ctx->b.items.p) + ub;
            a.nUnits = (int32_t)(ue - ub);
            a.queue = static_cast<uint32_t *>(ctx->b.queue.p) + c;
            a.rowbuf = static_cast<uint64_t *>(ctx->b.rowbuf.p);
            a.slotWords = slotWords;
            a.strips = static_cast<uint64_t *>(ctx->b.strips.p);
            a.stripWords = chunkStrips[c];
            a.error = ctx->waitFlag;
            a.mode = mode;
            a.alpha = A;
            a.tTable = static_cast<const int16_t *>(ctx->b.tTable.p);
            a.dnaProfile = static_cast<const uint32_t *>(ctx->b.dnaProf.p);
            a.drift = P.drift;
            a.trace = static_cast<uint4 *>(ctx->b.trace.p);
            a.traceRecs = traceRecs;
            a.traceOff = static_cast<const int64_t *>(ctx->b.traceOff.p) + b;
            a.ends = static_cast<TraceEnd *>(ctx->b.ends.p);
            a.endOff = static_cast<const int64_t *>(ctx->b.endOff.p) + b;
            if (chunkStrips[c] > 0 && (err = launchZero32(static_cast<uint32_t *>(ctx->b.strips.p),
                                                          2 * (size_t)chunkStrips[c], stream)) != hipSuccess)
                return hipFail(ctx, err, "launching fill kernel");
            const int cg = std::max(1, std::min(grid, (int)((ue - ub + wpb - 1) / wpb)));
            if ((err = launchTrace16(P.dna16, P.track, a, cg, stream)) != hipSuccess)
                return hipFail(ctx, err, "launching trace kernel");
            const int32_t p0 = tItems[b].first;
            const int32_t p1 = tItems[e - 1].first + tItems[e - 1].count;
            WalkArgs wa{};
            wa.hRes = in.dH;
            wa.vRes = in.dV;
            wa.hOff = a.hOff;
            wa.vOff = a.vOff;
            wa.ids = dOrder + p0;
            wa.locs = static_cast<const TraceLoc *>(ctx->b.locs.p) + p0;
            wa.nPairs = p1 - p0;
            wa.trace = a.trace;
            wa.ends = a.ends;
            wa.scores = in.dScores;
            wa.counts = dCounts;
            wa.alpha = A;
            wa.linear = si.o == si.e;
            wa.local = P.local ? 1 : 0;
            wa.table = static_cast<const int32_t *>(ctx->b.table32.p);
            wa.gapOpen = si.o;
            wa.gapExtend = si.e;
            wa.begins = rows.begins;
            wa.ops = rows.ops;
            wa.opOff = rows.opOff;
            wa.opLen = rows.opLen;
            if ((err = launchWalk16(wa, stream)) != hipSuccess)
                return hipFail(ctx, err, "launching walk kernel");
            b = e;
            ub = ue;
        }
    }
    // Banded pairs whose band, clipped to the matrix, has at most 512
    // diagonals: the lane-per-diagonal trace kernel (S trace bytes per row,
    // S = the widest band rounded up to a power of two), or up to 8 diagonals
    // per lane (S a multiple of 64), and a walk, in
    // chunks whose trace bytes fit the trace budget (offsets restart at 0 in
    // every chunk; the chunks run one after another on the call's stream).
    // SQMI_BANDED_TRACE_INT32=1 keeps them on the int32 kernel.
    int bandLanes = 0;
    std::vector<int64_t> bandOff;
    std::vector<size_t> bandChunkEnd;
    int64_t bandBytes = 0;
    if (band && !P.ids32.empty() && !envFlag("SQMI_BANDED_TRACE_INT32")) {
        int64_t wmax = 1;
        for (int32_t id : P.ids32) {
            const int64_t n = setH->offsets[id + 1] - setH->offsets[id], m = setV->offsets[id + 1] - setV->offsets[id];
            wmax = std::max(wmax, std::min(band[1], n) - std::max(band[0], -m) + 1);
        }
        if (wmax <= kMaxBandTrace) {
            bandLanes = 1;
            while (bandLanes < std::min<int64_t>(wmax, 64))
                bandLanes <<= 1;
            if (wmax > 64)
                bandLanes = (int)((wmax + 63) / 64 * 64);
            bandOff.resize(P.ids32.size());
            int64_t run = 0;
            for (size_t k = 0; k < P.ids32.size(); ++k) {
                const int32_t id = P.ids32[k];
                const int64_t need = (setV->offsets[id + 1] - setV->offsets[id]) * bandLanes;
                if (run > 0 && run + need > budget) {
                    bandChunkEnd.push_back(k);
                    run = 0;
                }
                bandOff[k] = run;
                run += need;
                bandBytes = std::max(bandBytes, run);
            }
            bandChunkEnd.push_back(P.ids32.size());
        }
    }
    if (bandLanes > 0) {
        const size_t n32 = P.ids32.size();
        if ((err = ensure(ctx->b.scratch32, (size_t)std::max<int64_t>(bandBytes, 1))) != hipSuccess ||
            (err = ensure(ctx->b.endEF, (size_t)8 * N)) != hipSuccess || (err = ensure(ctx->b.endIJ, (size_t)8 * N)) != hipSuccess)
            return hipFail(ctx, err, "allocating banded traceback buffers");
        if ((err = put(ctx, ctx->b.ids32, P.ids32.data(), 4 * n32)) != hipSuccess ||
            (err = put(ctx, ctx->b.scratchOff32, bandOff.data(), 8 * n32)) != hipSuccess || (err = stageFlush(ctx)) != hipSuccess)
            return hipFail(ctx, err, "uploading banded traceback lists");
        size_t cb = 0;
        for (size_t ce : bandChunkEnd) {
        BandedArgs ba{};
        ba.hRes = in.dH;
        ba.vRes = in.dV;
        ba.hOff = static_cast<const int64_t *>(ctx->b.hOff.p);
        ba.vOff = static_cast<const int64_t *>(ctx->b.vOff.p);
        ba.ids = static_cast<const int32_t *>(ctx->b.ids32.p) + cb;
        ba.nIds = (int32_t)(ce - cb);
        ba.scores = in.dScores;
        ba.gapOpen = si.o;
        ba.gapExtend = si.e;
        ba.mode = mode;
        ba.alpha = A;
        ba.table = static_cast<const int32_t *>(ctx->b.table32.p);
        ba.lower = band[0];
        ba.upper = band[1];
        ba.trace = static_cast<uint8_t *>(ctx->b.scratch32.p);
        ba.traceOff = static_cast<const int64_t *>(ctx->b.scratchOff32.p) + cb;
        ba.endIJ = static_cast<int32_t *>(ctx->b.endIJ.p);
        ba.endEF = static_cast<int32_t *>(ctx->b.endEF.p);
        if ((err = launchBandedTrace(ba, bandLanes, stream)) != hipSuccess)
            return hipFail(ctx, err, "launching banded trace kernel");
        BandedWalkArgs wa{};
        wa.hRes = in.dH;
        wa.vRes = in.dV;
        wa.hOff = ba.hOff;
        wa.vOff = ba.vOff;
        wa.ids = ba.ids;
        wa.nIds = ba.nIds;
        wa.segLanes = bandLanes;
        wa.lower = band[0];
        wa.upper = band[1];
        wa.trace = ba.trace;
        wa.traceOff = ba.traceOff;
        wa.scores = in.dScores;
        wa.endIJ = ba.endIJ;
        wa.endEF = ba.endEF;
        wa.counts = dCounts;
        wa.alpha = A;
        wa.local = (mode & SQMI_LOCAL) ? 1 : 0;
        wa.linear = si.o == si.e;
        wa.ops = rows.ops;
        wa.opOff = rows.opOff;
        wa.opLen = rows.opLen;
        wa.begins = rows.begins;
        if ((err = launchBandedWalk(wa, stream)) != hipSuccess)
            return hipFail(ctx, err, "launching banded walk kernel");
        cb = ce;
        }
    } else if (!P.ids32.empty()) {
        const size_t n32 = P.ids32.size();
        if ((err = ensure(ctx->b.scratch32, (size_t)scratch32)) != hipSuccess)
            return hipFail(ctx, err, "allocating int32 traceback buffers");
        if ((err = put(ctx, ctx->b.ids32, P.ids32.data(), 4 * n32)) != hipSuccess ||
            (err = put(ctx, ctx->b.scratchOff32, off32.data(), 8 * n32)) != hipSuccess || (err = stageFlush(ctx)) != hipSuccess)
            return hipFail(ctx, err, "uploading int32 traceback lists");
        size_t b = 0;
        for (size_t e : chunk32End) {
            Counts32Args a{};
            a.hRes = in.dH;
            a.vRes = in.dV;
            a.hOff = static_cast<const int64_t *>(ctx->b.hOff.p);
            a.vOff = static_cast<const int64_t *>(ctx->b.vOff.p);
            a.ids = static_cast<const int32_t *>(ctx->b.ids32.p) + b;
            a.scratchOff = static_cast<const int64_t *>(ctx->b.scratchOff32.p) + b;
            a.nIds = (int32_t)(e - b);
            a.scratch = static_cast<uint8_t *>(ctx->b.scratch32.p);
            a.scores = in.dScores;
            a.counts = dCounts;
            a.gapOpen = si.o;
            a.gapExtend = si.e;
            a.mode = mode;
            a.alpha = A;
            a.table = static_cast<const int32_t *>(ctx->b.table32.p);
            a.ops = rows.ops;
            a.opOff = rows.opOff;
            a.opLen = rows.opLen;
            a.begins = rows.begins;
            if (band) {
                a.banded = 1;
                a.lower = band[0];
                a.upper = band[1];
            }
            if ((err = launchCounts32(a, stream)) != hipSuccess)
                return hipFail(ctx, err, "launching int32 traceback kernel");
            b = e;
        }
    }
    if ((err = stageFlush(ctx)) != hipSuccess)   // offsets and tables, where no list above sent them
        return hipFail(ctx, err, "uploading");
    LongStage longStage;
    if ((st = runLong(ctx, setH, setV, P, in, flags, dCounts, rows, longStage)) != SQMI_OK)
        return st;
    if (!P.emptyIds.empty()) {
        if ((err = ensure(ctx->b.emptyIds, 4 * P.emptyIds.size())) != hipSuccess)
            return hipFail(ctx, err, "allocating empty list");
        if ((err = hipMemcpyAsync(ctx->b.emptyIds.p, P.emptyIds.data(), 4 * P.emptyIds.size(), hipMemcpyHostToDevice,
                                  stream)) != hipSuccess)
            return hipFail(ctx, err, "uploading empty list");
        if ((err = launchFillScores(in.dScores, static_cast<const int32_t *>(ctx->b.emptyIds.p), (int)P.emptyIds.size(),
                                    INT32_MIN, stream)) != hipSuccess)
            return hipFail(ctx, err, "launching fill kernel");
    }
    const uint8_t *rowsOut = rows.ops;
    if (wantRows && (flags & SQMI_ROWS_PACKED)) {
        // Rows back to back in pair order from ops + op_offsets[0].
        const int64_t opBytes = opOffsets[N];
        if ((err = ensure(ctx->b.opsPacked, (size_t)std::max<int64_t>(opBytes, 1))) != hipSuccess ||
            (err = ensure(ctx->b.opStart, 8 * (N + 1))) != hipSuccess)
            return hipFail(ctx, err, "allocating packed rows");
        uint8_t *packed = static_cast<uint8_t *>(ctx->b.opsPacked.p);
        if ((err = launchPackRows(rows.ops, rows.opOff, rows.opLen, static_cast<int64_t *>(ctx->b.opStart.p), packed,
                                  N, stream)) != hipSuccess)
            return hipFail(ctx, err, "launching row packing");
        if ((flags & SQMI_SCORES_ON_DEVICE) &&
            (err = hipMemcpyAsync(ops + opOffsets[0], packed + opOffsets[0], (size_t)(opBytes - opOffsets[0]),
                                  hipMemcpyDeviceToDevice, stream)) != hipSuccess)
            return hipFail(ctx, err, "copying packed rows");
        rowsOut = packed;
    }
    if ((err = hipEventRecord(ctx->ev1, stream)) != hipSuccess)
        return hipFail(ctx, err, "event");
    if (!(flags & SQMI_SCORES_ON_DEVICE)) {
        if ((err = fetch(ctx, scores, in.dScores, 4 * N)) != hipSuccess ||
            (err = fetch(ctx, counts, dCounts, (size_t)4 * S * N)) != hipSuccess)
            return hipFail(ctx, err, "copying results");
        if (wantRows && ((err = fetch(ctx, opLengths, rows.opLen, 8 * N)) != hipSuccess ||
                         (begins && (err = fetch(ctx, begins, rows.begins, 16 * N)) != hipSuccess)))
            return hipFail(ctx, err, "copying rows");
        if (wantRows) {
            // Packed rows fill only the first sum(op_lengths) bytes: read
            // that total (the scan's last entry) and copy no more.
            int64_t opsBytes = opOffsets[N] - opOffsets[0];
            size_t early = 0;   // results that have arrived with the total
            if (flags & SQMI_ROWS_PACKED) {
                int64_t total = 0;
                early = ctx->down.size();
                if ((err = fetch(ctx, &total, static_cast<const int64_t *>(ctx->b.opStart.p) + N, 8)) != hipSuccess ||
                    (err = hipStreamSynchronize(stream)) != hipSuccess)
                    return hipFail(ctx, err, "reading the packed rows' length");
                if (ctx->down.size() > early) {
                    std::memcpy(&total, ctx->down.back().src, 8);
                    ctx->down.pop_back();
                }
                opsBytes = std::min(opsBytes, std::max<int64_t>(total, 0));
            }
            if (opsBytes > 0 && (err = fetch(ctx, ops + opOffsets[0], rowsOut + opOffsets[0], (size_t)opsBytes)) != hipSuccess)
                return hipFail(ctx, err, "copying rows");
            deliver(ctx, early);   // while the rows are on their way
        }
    }
    if ((err = hipStreamSynchronize(stream)) != hipSuccess)
        return hipFail(ctx, err, "traceback kernels");
    deliver(ctx);
    stageEnd(ctx);
    if ((st = stripCheck(ctx)) != SQMI_OK)
        return st;
    float ms = 0;
    if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) == hipSuccess)
        ctx->stats.device_ms = ms;
    ctx->stats.total_ms = msSince(tStart);
    return SQMI_OK;
}

sqmi_status sqmi_align_counts(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                              const sqmi_scoring *scoring, uint32_t mode, int32_t *scores, int32_t *counts,
                              uint32_t flags)
{
    return alignBackward(ctx, setH, setV, scoring, mode, scores, counts, nullptr, nullptr, nullptr, nullptr, flags);
}

sqmi_status sqmi_align_rows(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                            const sqmi_scoring *scoring, uint32_t mode, int32_t *scores, int32_t *counts,
                            uint8_t *ops, const int64_t *op_offsets, int64_t *op_lengths, uint32_t flags)
{
    if (!ops)
        return ctx ? fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "ops is null") : SQMI_ERR_INVALID_ARGUMENT;
    if (mode & SQMI_LOCAL)
        return ctx ? fail(ctx, SQMI_ERR_UNSUPPORTED,
                          "sqmi_align_rows: global modes only; local rows come from sqmi_align_local_rows")
                   : SQMI_ERR_UNSUPPORTED;
    return alignBackward(ctx, setH, setV, scoring, mode, scores, counts, ops, op_offsets, op_lengths, nullptr, flags);
}

// Bands the library computes: the band holds the diagonals of (0, 0) and of
// (m, n) with at least one more diagonal beyond each, and H has at least two
// residues.  There the reference's banded code computes the banded
// recurrence.  Elsewhere it takes special paths of its own
// (dp_algorithm_impl.h:595-700: one-diagonal bands, single-column matrices,
// bands whose edge lies on a corner diagonal) whose results differ from that
// recurrence under free end gaps or for |H| = 1, so such requests are
// refused.  Without free ends the reference itself accepts only bands that
// hold both corners (_checkBandProperties, dp_algorithm_impl.h:192-232).
//
// Local alignment (every end free): |H| >= 2, at least two diagonals, and
// the band reaches past the corner cells (0, n - 1) and (m - 1, 0): bands
// that only touch a corner, or have one diagonal, again take the special
// paths.
static bool bandSupported(int64_t n, int64_t m, int64_t lower, int64_t upper, bool local)
{
    if (local)
        return n >= 2 && lower < upper && lower <= n - 2 && upper >= -(m - 2) &&
               std::min<int64_t>(upper, n) - std::max<int64_t>(lower, -m) >= 1;
    return n >= 2 && lower < std::min<int64_t>(0, n - m) && upper > std::max<int64_t>(0, n - m);
}

sqmi_status sqmi_align_score_banded(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                                    const sqmi_scoring *scoring, uint32_t mode, int64_t lower_diag,
                                    int64_t upper_diag, int32_t *scores, uint32_t flags)
{
    const auto tStart = std::chrono::steady_clock::now();
    if (!ctx)
        return SQMI_ERR_INVALID_ARGUMENT;
    dropReplay(ctx);   // this call rewrites the buffers a replay would reuse
    ctx->lastError.clear();
    ctx->stats = sqmi_stats{};
    sqmi_status st;
    if ((st = validate(ctx, setH, setV, scoring, mode)) != SQMI_OK)
        return st;
    const bool local = (mode & SQMI_LOCAL) != 0;
    if (flags & ~(uint32_t)(SQMI_RESIDUES_ON_DEVICE | SQMI_SCORES_ON_DEVICE | SQMI_FORCE_INT32))
        return fail(ctx, SQMI_ERR_UNSUPPORTED,
                    "sqmi_align_score_banded: flags other than the *_ON_DEVICE ones and SQMI_FORCE_INT32");
    if (lower_diag > upper_diag)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "lower_diag > upper_diag");
    const int64_t N = setH->count;
    if (N == 0)
        return SQMI_OK;
    if (!scores)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "scores is null");
    if (hipSetDevice(ctx->device) != hipSuccess)
        return fail(ctx, SQMI_ERR_DEVICE, "hipSetDevice failed");
    hipStream_t stream = ctx->stream;

    // Large host residue sets are copied in on a second host thread while
    // this one routes the pairs (as in the rows calls).
    Inputs in;
    hipError_t upErr = hipSuccess;
    JoinedThread up;
    if (!(flags & SQMI_RESIDUES_ON_DEVICE) && setH->offsets[N] + setV->offsets[N] >= ((int64_t)4 << 20))
        up.t = std::thread([&] {
            upErr = hipSetDevice(ctx->device);
            if (upErr == hipSuccess)
                upErr = uploadResidues(ctx, setH, setV, in);
        });

    // Route: empty pairs (INT32_MIN), the packed int16 kernel (values inside
    // 16 bits, at least 8 diagonals past the first), narrow bands (<= 64
    // diagonals), wide bands.
    const auto tPlan = std::chrono::steady_clock::now();
    ScoringInfo si{};
    si.alpha = scoring->alphabet_size;
    si.o = scoring->gap_open;
    si.e = scoring->gap_extend;
    si.sMax = INT_MIN;
    si.sMin = INT_MAX;
    for (int k = 0; k < si.alpha * si.alpha; ++k) {
        si.sMax = std::max(si.sMax, scoring->table[k]);
        si.sMin = std::min(si.sMin, scoring->table[k]);
    }
    si.dna = si.alpha <= 4 && si.sMin - si.o >= 0 && si.sMax - si.o <= 255;
    const int64_t W1 = upper_diag - lower_diag;
    // Rows per block: more rows share a block's set-up and boundary columns,
    // fewer compute fewer cells outside the band (W - 1 + R columns per
    // block for W band cells per row).  In plain values, a wave per item: band
    // [-16, 16] on 1 M pairs of 150 bp: R = 12 1.64 ms, 16 1.74 ms; [-100,
    // 100] on 65,536 pairs of 1 kbp: R = 16 4.66 ms, 12 5.10 ms.
    const int bandR = W1 >= 64 ? 16 : W1 >= 24 ? 12 : 8;
    si.dnaDrift = si.dna && si.sMax - si.o - std::max(si.o, si.e) <= 255;
    const bool bandCostsOk = !(flags & SQMI_FORCE_INT32) && W1 >= bandR && si.o <= 0 && si.e <= 0 && si.o >= -1024 &&
                             si.e >= -1024 && si.sMax <= 1024 && si.sMin >= -1024 && si.alpha + 1 <= 33 &&
                             lower_diag > -30000 && upper_diag < 30000;
    // The packed kernel's values: the bias covers the longest pair of the
    // call; columns run to the item's longest |H|, a group past the band.
    Drift dr = driftOf(si, local);
    const int64_t *offH = setH->offsets, *offV = setV->offsets;
    int64_t maxN = 1, maxM = 1, nTop = 1;   // nTop: |H| of a pair of the most rows (calls of one thread)
    if (N > kParallelMin) {
#pragma omp parallel for schedule(static) reduction(max : maxN, maxM)
        for (int64_t i = 0; i < N; ++i) {
            maxN = std::max(maxN, offH[i + 1] - offH[i]);
            maxM = std::max(maxM, offV[i + 1] - offV[i]);
        }
    } else if (bandCostsOk) {
        for (int64_t i = 0; i < N; ++i) {
            const int64_t n = offH[i + 1] - offH[i], m = offV[i + 1] - offV[i];
            maxN = std::max(maxN, n);
            nTop = m > maxM ? n : nTop;
            maxM = std::max(maxM, m);
        }
    }
    if (!local && bandCostsOk)
        dr.bias += (int32_t)std::min<int64_t>(bandDrop(si, dr, W1, maxM), 1 << 20);
    auto bandTop = [&](int64_t m) {   // the largest stored value of pairs with m rows
        const int64_t cols = std::min(maxN, m + upper_diag) + 8;
        return dr.bias + (int64_t)std::max(si.sMax, 0) * std::min(m, cols) + dr.d * (local ? 17 : m + cols);
    };
    const bool narrowT = dr.neg == (local ? 2 * dr.d + 2 : dr.cost + 1);   // no t below 0
    bool bandWide = !narrowT;
    // Free end gaps and local alignment, few pairs: a packed item takes its
    // whole sweep, however few the items; the int32 kernels, which spread a
    // pair's band over a wave, are done earlier.  Times in ns: a call's items
    // on the packed kernel, a pair on int32 (alone; its share of a full chip).
    const double simds = 4.0 * std::max(1, ctx->numCUs);
    auto packedTime = [&](double items, double blockCols, int64_t most) {
        const int cols = bandRingCols((int)most, lower_diag, upper_diag, bandR), waves = bandWaves(cols);
        const double slots = cols > 256 ? simds : 2 * simds / waves;
        const double column = cols > 256 ? kBandColumnAlone : kBandColumn[waves == 8 ? 2 : waves == 4 ? 1 : 0];
        return std::ceil(items / slots) * blockCols * column;
    };
    auto loneTime = [&](double m, double w) { return m * (w <= 64 ? kBandNarrowLone : kBandWideLone * std::ceil(w / 64)); };
    auto fullTime = [&](double m, double w) {
        return m * (w <= 64 ? kBandNarrowFull * w / 64 : kBandWideFull * std::ceil(w / 64)) / simds;
    };
    const bool choose = mode != 0 && !envFlag("SQMI_BAND_PACKED");
    bool packedOk = bandCostsOk;
    if (choose && packedOk && N <= kParallelMin && maxN <= 30000 && maxM <= 30000) {
        // From the sums alone, where the least that the packed kernel takes
        // (the tallest pair's item) exceeds the most that int32 does: the
        // pairs need not be placed first (20,000 pairs of 1 kbp, 11 diagonals,
        // local: a call 0.69 -> 0.54 ms).
        const double w = std::min<double>((double)W1 + 1, (double)(maxN + maxM));
        const double wTop = std::min<double>((double)W1 + 1, (double)(nTop + maxM));
        const double blockCols = ((maxM + bandR) / bandR) * std::min<double>(wTop + bandR, (double)nTop);
        packedOk = std::max(loneTime((double)maxM, w), fullTime((double)(offV[N] - offV[0]), w)) >=
                   packedTime(std::ceil((double)N / 128), blockCols, nTop);
    }
    std::vector<int32_t> narrow, wide, rejected;
    int64_t wNarrow = 1, wWide = 0, cells = 0;
    auto toInt32 = [&](int32_t id, int64_t n, int64_t m) {
        const int64_t w = std::min<int64_t>(upper_diag, n) - std::max<int64_t>(lower_diag, -m) + 1;
        if (w <= 64) {
            narrow.push_back(id);
            wNarrow = std::max(wNarrow, w);
        } else {
            wide.push_back(id);
            wWide = std::max(wWide, w);
        }
    };
    // Every thread routes a contiguous part of the pairs and counts its packed
    // pairs by |V|; the counts' prefix sums (by |V|, then thread) place them,
    // in pair order within a |V|.  On 1,048,576 pairs one thread took 5 ms.
    auto packs = [&](int64_t n, int64_t m) { return packedOk && n <= 30000 && m <= 30000 && bandTop(m) <= 65535; };
    const int64_t mSlots = std::min<int64_t>(maxM, 30000) + 1;
    const int parts = N > kParallelMin ? (int)std::max<int64_t>(1, std::min<int64_t>(omp_get_max_threads(), N / mSlots)) : 1;
    std::vector<int32_t> counts((size_t)parts * mSlots, 0);
    std::vector<int64_t> nOther((size_t)parts, 0);
    int64_t firstBad = N, nPacked = 0;
    bool anyWide = false;
    const bool routed = !packedOk && parts == 1;   // one pass: no pair is packed
    if (routed) {
        narrow.reserve((size_t)N);
        for (int64_t i = 0; i < N && firstBad == N; ++i) {
            const int64_t n = offH[i + 1] - offH[i], m = offV[i + 1] - offV[i];
            if (n == 0 || m == 0) {
                rejected.push_back((int32_t)i);
            } else if (!bandSupported(n, m, lower_diag, upper_diag, local)) {
                firstBad = i;
            } else {
                cells += n * m;
                toInt32((int32_t)i, n, m);
            }
        }
    }
#pragma omp parallel for schedule(static) num_threads(parts) reduction(+ : cells, nPacked) reduction(min : firstBad) \
    reduction(|| : anyWide) if (parts > 1)
    for (int t = 0; t < parts; ++t) {
        int32_t *cnt = counts.data() + (size_t)t * mSlots;
        for (int64_t i = N * t / parts; i < N * (t + 1) / parts && !routed; ++i) {
            const int64_t n = offH[i + 1] - offH[i], m = offV[i + 1] - offV[i];
            if (n != 0 && m != 0 && !bandSupported(n, m, lower_diag, upper_diag, local)) {
                firstBad = std::min(firstBad, i);
                continue;
            }
            cells += n != 0 && m != 0 ? n * m : 0;
            if (n != 0 && m != 0 && packs(n, m)) {
                ++cnt[m];
                ++nPacked;
                anyWide = anyWide || bandTop(m) > kDriftNarrowMax;
            } else {
                ++nOther[(size_t)t];
            }
        }
    }
    if (firstBad < N)
        return fail(ctx, SQMI_ERR_UNSUPPORTED,
                    "sqmi_align_score_banded: pair " + std::to_string(firstBad) +
                        (local ? ": needs |H| >= 2, two diagonals, lower_diag <= |H| - 2 and upper_diag >= 2 - |V|"
                               : ": needs |H| >= 2 and lower_diag < min(0, |H| - |V|) < max(0, |H| - |V|) "
                                 "< upper_diag"));
    bandWide |= anyWide;
    for (int t = 0; t < parts; ++t)
        for (int64_t i = N * t / parts; nOther[(size_t)t] > 0 && i < N * (t + 1) / parts; ++i) {
            const int64_t n = offH[i + 1] - offH[i], m = offV[i + 1] - offV[i];
            if (n == 0 || m == 0)
                rejected.push_back((int32_t)i);
            else if (!packs(n, m))
                toInt32((int32_t)i, n, m);
        }
    // Packed items: up to 128 pairs of one |V|.
    RawVec<int32_t> packed((size_t)nPacked);
    std::vector<WorkItem> bandItems;
    int bandMaxN = 1;
    if (nPacked > 0) {
        int32_t run = 0;
        for (int64_t mm = 0; mm < mSlots; ++mm) {
            const int32_t f0 = run;
            for (int t = 0; t < parts; ++t) {
                int32_t &c = counts[(size_t)t * mSlots + mm];
                const int32_t k = c;
                c = run;
                run += k;
            }
            for (int32_t f = f0; f < run; f += 128)
                bandItems.push_back(WorkItem{f, std::min<int32_t>(128, run - f) | ((int)mm << 16), 1,
                                             ((int)mm + bandR) / bandR});
        }
#pragma omp parallel for schedule(static) num_threads(parts) if (parts > 1)
        for (int t = 0; t < parts; ++t) {
            int32_t *pos = counts.data() + (size_t)t * mSlots;
            for (int64_t i = N * t / parts; i < N * (t + 1) / parts; ++i) {
                const int64_t n = offH[i + 1] - offH[i], m = offV[i + 1] - offV[i];
                if (n != 0 && m != 0 && packs(n, m))
                    packed[(size_t)pos[m]++] = (int32_t)i;
            }
        }
#pragma omp parallel for schedule(static) reduction(max : bandMaxN) if (parts > 1)
        for (int64_t k = 0; k < (int64_t)bandItems.size(); ++k) {
            WorkItem &w = bandItems[(size_t)k];
            for (int32_t q = w.first; q < w.first + (w.count & 0xffff); ++q)
                w.maxN = std::max(w.maxN, (int)(offH[packed[q] + 1] - offH[packed[q]]));
            bandMaxN = std::max(bandMaxN, w.maxN);
        }
    }
    if (choose && !packed.empty()) {
        double blockCols = 0, lone = 0, full = 0;
        for (const WorkItem &it : bandItems) {
            const double m = (double)((uint32_t)it.count >> 16), w = std::min<double>((double)W1 + 1, it.maxN + m);
            blockCols = std::max(blockCols, it.nblocks * std::min<double>(w + bandR, it.maxN));
            lone = std::max(lone, loneTime(m, w));
            full += (it.count & 0xffff) * fullTime(m, w);
        }
        if (std::max(lone, full) < packedTime((double)bandItems.size(), blockCols, bandMaxN)) {
            for (int32_t id : packed)
                toInt32(id, offH[id + 1] - offH[id], offV[id + 1] - offV[id]);
            packed.clear();
            bandItems.clear();
        }
    }
    int seg = 1;
    while (seg < wNarrow)
        seg <<= 1;
    ctx->stats.pairs = N;
    ctx->stats.cells = cells;
    ctx->stats.pairs_int32 = (int64_t)(narrow.size() + wide.size());
    ctx->stats.pairs_int16 = (int64_t)packed.size();
    ctx->stats.host_plan_ms = msSince(tPlan);

    up.join();
    if (upErr != hipSuccess)
        return hipFail(ctx, upErr, "copying residues");
    hipError_t err;
    if ((err = stageBegin(ctx, stageInputs(setH, setV, scoring, flags) + stageBytes(4 * (size_t)N) + stageBytes(4 * packed.size()) +
                                   stageBytes(sizeof(WorkItem) * bandItems.size()) + 1024,
                          downScores(N, flags))) != hipSuccess)
        return hipFail(ctx, err, "allocating upload staging");
    if ((st = uploadInputs(ctx, setH, setV, scoring, si, scores, flags, in)) != SQMI_OK)
        return st;
    const int wideStride = (int)((wWide + 2 + 63) & ~(int64_t)63);
    const int wideGrid = wide.empty() ? 0 : (int)std::min<int64_t>((int64_t)wide.size(), (int64_t)ctx->numCUs * 16);
    const size_t nIds = narrow.size() + wide.size() + rejected.size();
    if ((wideGrid && (err = ensure(ctx->b.bandScratch, (size_t)wideGrid * 4 * wideStride * 4)) != hipSuccess))
        return hipFail(ctx, err, "allocating banded buffers");
    std::vector<int32_t> all(narrow);
    all.insert(all.end(), wide.begin(), wide.end());
    all.insert(all.end(), rejected.begin(), rejected.end());
    if ((err = put(ctx, ctx->b.bandIds, all.data(), 4 * nIds)) != hipSuccess)
        return hipFail(ctx, err, "uploading banded pair lists");
    int32_t *dIds = static_cast<int32_t *>(ctx->b.bandIds.p);
    int bandGrid = 0, bandRowColsN = 0, bandLds = 0;
    BandVariant bandVar{};
    if (!bandItems.empty()) {
        // Rings of up to 256 columns (128 KB) live in LDS, one per workgroup,
        // whose waves share an item; 8 waves per CU whatever the ring.
        // Larger ones lie in global memory, one per wave: as many workgroups
        // of 4 waves as keep a CU's rings within its share of L2 (at least
        // one; more send the rings to memory).
        bandRowColsN = bandRingCols(bandMaxN, lower_diag, upper_diag, bandR);
        bandLds = bandLdsRingBytes(bandRowColsN);
        // The DNA form keeps scores in bytes, also the one that holds row 0 at
        // H = 0 under a free first row: -gapOpen, which only schemes whose
        // scores are all negative let past 255.  The table holds it in 16 bits.
        const bool padFits = !(mode & SQMI_FREE_TOP) || si.o >= -255;
        bandVar = BandVariant{bandR, padFits && (local ? si.dna : si.dnaDrift),
                              local ? kBandLocal : (mode & (SQMI_FREE_BOTTOM | SQMI_FREE_RIGHT)) ? kBandFree : kBandEnd,
                              bandWide, bandLds > 0, bandWaves(bandRowColsN)};
        const int64_t ringBytes = (int64_t)64 * bandRowColsN * 8;   // per wave
        const int most = occupancyBand16(bandVar, bandLds);
        const int occ = bandLds ? most : (int)std::max<int64_t>(1, std::min<int64_t>(most, ctx->l2PerCU / (4 * ringBytes)));
        const int64_t nIt = (int64_t)bandItems.size();
        bandGrid = std::max(1, (int)std::min<int64_t>((int64_t)ctx->numCUs * occ, bandLds ? nIt : (nIt + 3) / 4));
        if ((err = ensure(ctx->b.queue, 64)) != hipSuccess ||
            (err = ensure(ctx->b.rowbuf, bandLds ? 64 : (size_t)bandGrid * 4 * 64 * bandRowColsN * 8)) != hipSuccess)
            return hipFail(ctx, err, "allocating packed banded buffers");
        if ((err = put(ctx, ctx->b.order, packed.data(), 4 * packed.size())) != hipSuccess ||
            (err = put(ctx, ctx->b.items, bandItems.data(), sizeof(WorkItem) * bandItems.size())) != hipSuccess)
            return hipFail(ctx, err, "uploading packed banded work");
    }
    if ((err = stageFlush(ctx)) != hipSuccess)
        return hipFail(ctx, err, "uploading");
    if ((err = hipEventRecord(ctx->ev0, stream)) != hipSuccess)
        return hipFail(ctx, err, "event");
    if (!bandItems.empty()) {
        if ((err = launchZero32(static_cast<uint32_t *>(ctx->b.queue.p), 16, stream)) != hipSuccess)
            return hipFail(ctx, err, "launching queue reset");
        FwdArgs f{};
        f.hRes = in.dH;
        f.vRes = in.dV;
        f.hOff = static_cast<const int64_t *>(ctx->b.hOff.p);
        f.vOff = static_cast<const int64_t *>(ctx->b.vOff.p);
        f.order = static_cast<const int32_t *>(ctx->b.order.p);
        f.items = static_cast<const WorkItem *>(ctx->b.items.p);
        f.nItems = (int32_t)bandItems.size();
        f.queue = static_cast<uint32_t *>(ctx->b.queue.p);
        f.rowbuf = static_cast<uint32_t *>(ctx->b.rowbuf.p);
        f.rowCols = bandRowColsN;
        f.bandCols = bandRowColsN;
        f.scores = in.dScores;
        f.gapOpen = si.o;
        f.gapExtend = si.e;
        f.mode = mode;
        f.alpha = si.alpha;
        f.tTable = static_cast<const int16_t *>(ctx->b.tTable.p);
        f.dnaProfile = static_cast<const uint32_t *>(ctx->b.dnaProf.p);
        f.drift = dr;
        f.error = ctx->waitFlag;
        f.bandLo = (int32_t)lower_diag;
        f.bandUp = (int32_t)upper_diag;
        if ((err = launchBand16(bandVar, f, bandGrid, bandLds, stream)) != hipSuccess)
            return hipFail(ctx, err, "launching packed banded kernel");
    }
    BandedArgs a{};
    a.hRes = in.dH;
    a.vRes = in.dV;
    a.hOff = static_cast<const int64_t *>(ctx->b.hOff.p);
    a.vOff = static_cast<const int64_t *>(ctx->b.vOff.p);
    a.scores = in.dScores;
    a.gapOpen = si.o;
    a.gapExtend = si.e;
    a.mode = mode;
    a.alpha = si.alpha;
    a.table = static_cast<const int32_t *>(ctx->b.table32.p);
    a.lower = lower_diag;
    a.upper = upper_diag;
    a.scratch = static_cast<int32_t *>(ctx->b.bandScratch.p);
    a.wideStride = wideStride;
    if (!narrow.empty()) {
        a.ids = dIds;
        a.nIds = (int32_t)narrow.size();
        if ((err = launchBanded(a, seg, 0, stream)) != hipSuccess)
            return hipFail(ctx, err, "launching banded kernel");
    }
    if (!wide.empty()) {
        a.ids = dIds + narrow.size();
        a.nIds = (int32_t)wide.size();
        if ((err = launchBanded(a, 0, wideGrid, stream)) != hipSuccess)
            return hipFail(ctx, err, "launching banded kernel");
    }
    if (!rejected.empty() &&
        (err = launchFillScores(in.dScores, dIds + narrow.size() + wide.size(), (int)rejected.size(), INT32_MIN,
                                stream)) != hipSuccess)
        return hipFail(ctx, err, "launching fill kernel");
    if ((err = hipEventRecord(ctx->ev1, stream)) != hipSuccess)
        return hipFail(ctx, err, "event");
    if (!(flags & SQMI_SCORES_ON_DEVICE) && (err = fetch(ctx, scores, in.dScores, 4 * N)) != hipSuccess)
        return hipFail(ctx, err, "copying scores");
    if ((err = hipStreamSynchronize(stream)) != hipSuccess)
        return hipFail(ctx, err, "banded kernels");
    deliver(ctx);
    stageEnd(ctx);
    if ((st = stripCheck(ctx)) != SQMI_OK)
        return st;
    float ms = 0;
    if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) == hipSuccess)
        ctx->stats.device_ms = ms;
    ctx->stats.total_ms = msSince(tStart);
    return SQMI_OK;
}

sqmi_status sqmi_align_local_rows(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                                  const sqmi_scoring *scoring, int32_t *scores, int32_t *counts, uint8_t *ops,
                                  const int64_t *op_offsets, int64_t *op_lengths, int64_t *begins, uint32_t flags)
{
    if (!ops || !begins)
        return ctx ? fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "ops or begins is null") : SQMI_ERR_INVALID_ARGUMENT;
    return alignBackward(ctx, setH, setV, scoring, SQMI_LOCAL, scores, counts, ops, op_offsets, op_lengths, begins,
                         flags);
}

sqmi_status sqmi_align_rows_banded(sqmi_context *ctx, const sqmi_sequences *setH, const sqmi_sequences *setV,
                                   const sqmi_scoring *scoring, uint32_t mode, int64_t lower_diag,
                                   int64_t upper_diag, int32_t *scores, int32_t *counts, uint8_t *ops,
                                   const int64_t *op_offsets, int64_t *op_lengths, int64_t *begins, uint32_t flags)
{
    if (!ctx)
        return SQMI_ERR_INVALID_ARGUMENT;
    ctx->lastError.clear();
    sqmi_status st;
    if ((st = validate(ctx, setH, setV, scoring, mode)) != SQMI_OK)
        return st;
    if (flags & ~(uint32_t)(SQMI_RESIDUES_ON_DEVICE | SQMI_SCORES_ON_DEVICE | SQMI_ROWS_PACKED))
        return fail(ctx, SQMI_ERR_UNSUPPORTED,
                    "sqmi_align_rows_banded: flags other than the *_ON_DEVICE ones and SQMI_ROWS_PACKED");
    if (lower_diag > upper_diag)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "lower_diag > upper_diag");
    const bool local = (mode & SQMI_LOCAL) != 0;
    if (local && ops && !begins)
        return fail(ctx, SQMI_ERR_INVALID_ARGUMENT, "begins is null");
    for (int64_t i = 0; i < setH->count; ++i) {
        const int64_t n = setH->offsets[i + 1] - setH->offsets[i], m = setV->offsets[i + 1] - setV->offsets[i];
        if (n != 0 && m != 0 && !bandSupported(n, m, lower_diag, upper_diag, local))
            return fail(ctx, SQMI_ERR_UNSUPPORTED,
                        "sqmi_align_rows_banded: pair " + std::to_string(i) + " is outside the supported bands");
    }
    const int64_t band[2] = {lower_diag, upper_diag};
    return alignBackward(ctx, setH, setV, scoring, local ? (uint32_t)SQMI_LOCAL : mode, scores, counts, ops,
                         op_offsets, op_lengths, local ? begins : nullptr, flags, band);
}

}  // extern "C"
