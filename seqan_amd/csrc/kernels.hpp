// kernels.hpp -- interface between the host planner (engine.cpp) and the
// gfx950 kernels (kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace sqmi {

// Sentinel for "minus infinity" inside the packed int16 kernels.  Every real
// value of a pair routed to them is proven (on the host) to stay within
// [kNeg16 + kGuard16, 32767 - kGuard16].
constexpr int kNeg16 = -28672;
// Substitution tables of the packed forward: at most this many codes
// (alphabet + padding code) per side, held in LDS replicated per bank.
constexpr int kTabMaxCodes = 28;
constexpr int kGuard16 = 2048;

// Tracking kinds (which cells define the result), from the mode bits.
enum Track : uint32_t {
    kTrackEnd = 1,      // global: cell (m, n)
    kTrackBottom = 2,   // last row free: max over row m, j <= n
    kTrackRight = 4,    // last column free: max over column n, i <= m
    kTrackLocal = 8,    // local: max over all cells
    // Kernel variant flag of the one-pair-per-lane kernels (drifted values):
    // the values need all 16 bits (Variant16::wide).
    kWideVals = 32
};

// The global score kernels (packed, every AlignConfig) hold drifted values
// (the local ones drift along the sweep only, score16.hpp):
//   stored(i, j) = value(i, j) + drift * (i + j) + bias,   drift = -max(e, o)
// (extending past max(e, o) is never better than reopening, so max(e, o)
// stands for e).  A gap extension is then a step without cost, so
//   E = max(E, G), F = max(F, G), H = max(G(i-1,j-1) + t, E, F), G = H - cost
// with cost = max(e, o) - o and t = s + cost + 2 drift: five operations and
// the score lookup per cell instead of eight.  Every stored value is >= 0:
// `neg` stands for minus infinity, and no operation on a value >= neg gives a
// value below 1 (E never falls below neg, G not below neg - cost, a
// diagonal not below neg - cost + min t).  True values are at least bias -
// 3 cost (the all-gap path) and above neg.
struct Drift {
    int32_t d, cost, neg, bias;
};
// Stored values of at most this take the three-operand packed maximum
// (v_pk_maximum3_f16: as bit patterns, non-negative finite halves order like
// integers) and 32-bit sums and differences of both halves at once; above,
// up to 65535, unsigned packed maxima, sums and differences (kWideVals).
constexpr int kDriftNarrowMax = 0x7bff;
// Rows and columns past a pair's own that its item may sweep with real
// residues (one-pair-per-lane kernels): pairs of an item differ by less than
// a row block in |V|, and columns are swept in groups of 4.
constexpr int kDriftSlack = 64;

// A work item: up to `pairs per wave` pairs that share the same number of
// row blocks; processed together by one wavefront.
struct WorkItem {
    int32_t first;      // index of the first pair in `order`
    int32_t count;      // bits 0..15: number of pairs in the item; bits 16..17
                        // (packed kernels with G = 16 / 64): quarters of a block
                        // held by block 0 (0: a whole block); banded kernels:
                        // bits 16..31 the pairs' common |V|
    int32_t maxN;       // max |H| over the item's pairs
    int32_t nblocks;    // row blocks of G*R rows (same for all pairs)
};

struct FwdArgs {
    const uint8_t *hRes;
    const uint8_t *vRes;
    const int64_t *hOff;
    const int64_t *vOff;
    const int32_t *order;       // pair ids grouped by work item
    const WorkItem *items;
    int32_t nItems;
    uint32_t *queue;            // work-queue counter of the per-wave items (zeroed before launch)
    uint32_t *rowbuf;           // per wave slot: GROUPS * rowCols * 2 dwords
    int32_t rowCols;            // columns per group row buffer
    int32_t *scores;            // indexed by pair id
    int32_t gapOpen;
    int32_t gapExtend;
    uint32_t mode;              // SQMI_* mode bits
    int32_t alpha;              // alphabet size; residue code `alpha` is padding
    const int16_t *tTable;      // (alpha+1)^2 entries: s(h,v) - gapOpen, pad row/col
    const uint32_t *dnaProfile; // dwords 0..4: bytes v=0..3 of s(h,v)-gapOpen, h=0..3, pad;
                                // dwords 8..12: bytes h=0..3 of s(h,v)-gapOpen, v=0..3, pad
    Drift drift;                // global score kernels
    int32_t bandLo, bandUp;     // banded kernels: cells with bandLo <= j - i <= bandUp
    int32_t bandCols;           // banded kernels: row-buffer ring columns (a power of two <= rowCols)
    uint32_t *error;            // banded kernels: as in ScoreArgs
};

// Where the trace records of one pair live: rows are bottom-aligned in the
// item's blocks of 256 rows (row i is item row p + i), lane group lane0..+15,
// pair A or B (`half`) of the record's byte layout.
struct TraceLoc {
    int64_t rec0;               // first record of the item (units of 64 records)
    int32_t steps;              // column steps per block
    int32_t p;                  // item row of the pair's row 0
    int32_t lane0;              // first lane of the pair's group
    int32_t half;               // 0: low int16 half, 1: high
    int32_t lanes;              // lanes per couple: 16, or 64 (records of one word)
    // The end-cell candidates of the pair's units (strips of the item, or the
    // whole item): ends[end0 + q * endStride], q < nEnds.
    int64_t end0;
    int32_t endStride;
    int32_t nEnds;
    int32_t pad;
};

// End-cell candidates a trace unit leaves per pair, values in H: b, the best
// cell of the bottom row (global; only the last unit's counts) or of all its
// cells (local, none: j = INT32_MAX); r, the best cell of column n (free last
// column).
struct TraceEnd {
    int32_t v, i, j, e, f;
    int32_t rv, ri, rj, re, rf;
};

// Traceback walk: 16 lanes per pair, or a whole wave in calls of few pairs.
struct WalkArgs {
    const uint8_t *hRes;
    const uint8_t *vRes;
    const int64_t *hOff;
    const int64_t *vOff;
    const int32_t *ids;         // pair ids
    const TraceLoc *locs;       // per id
    int32_t nPairs;
    const uint4 *trace;
    const TraceEnd *ends;       // end-cell candidates (TraceLoc::end0)
    int32_t *scores;            // per pair id (output)
    int32_t *counts;            // per pair id: alpha^2 + 2 counts
    int32_t alpha;
    int32_t linear;             // gap open == gap extend: the linear-gap walk
    int32_t local;              // local walk: stops where H falls to 0, no leading / trailing gaps
    const int32_t *table;       // local: alpha^2 substitution scores (H along the path)
    int32_t gapOpen;
    int32_t gapExtend;
    int64_t *begins;            // local: per pair id, the window's first H and V position (optional)
    // Rows (optional): pair id p's ops end at ops[opOff[p + 1]] (written
    // backwards), their number goes to opLen[p].
    uint8_t *ops;
    const int64_t *opOff;
    int64_t *opLen;
};

// int32 traceback, one thread per pair, trace bytes in global scratch.
struct Counts32Args {
    const uint8_t *hRes;
    const uint8_t *vRes;
    const int64_t *hOff;
    const int64_t *vOff;
    const int32_t *ids;
    const int64_t *scratchOff;  // per thread: byte offset of its scratch
    int32_t nIds;
    uint8_t *scratch;           // 8 (m+1) bytes of H/E columns + (n+1)(m+1) trace bytes per pair
    int32_t *scores;
    int32_t *counts;
    int32_t gapOpen;
    int32_t gapExtend;
    uint32_t mode;              // free end gaps (SQMI_FREE_*) or SQMI_LOCAL
    int32_t alpha;
    const int32_t *table;
    uint8_t *ops;               // rows, as in WalkArgs (optional)
    const int64_t *opOff;
    int64_t *opLen;
    int64_t *begins;            // local: per pair the window's first H and V position (optional)
    int32_t banded;             // cells outside lower <= j - i <= upper are -inf
    int64_t lower;
    int64_t upper;
};

// Simple int32 kernel: one thread per pair, H/E column in global scratch.
struct Simple32Args {
    const uint8_t *hRes;
    const uint8_t *vRes;
    const int64_t *hOff;
    const int64_t *vOff;
    const int32_t *ids;         // pair ids
    const int64_t *scratchOff;  // per id slot: offset (in int32 pairs) of its column
    int32_t nIds;
    int32_t *scratch;           // 2 * (m+1) int32 per pair
    int32_t *scores;
    int32_t gapOpen;
    int32_t gapExtend;
    uint32_t mode;
    int32_t alpha;
    const int32_t *table;       // alpha^2 substitution scores
};

// The packed score kernels (score16.hpp).  Kinds: global modes without a free
// last column, with one, local.
enum ScoreKind : int { kScoreGlobal = 0, kScoreRight = 1, kScoreLocal = 2 };
// A unit of work: all row blocks of an item (block < 0), or one of them (a
// strip).  Up to 2 * 64 / G pairs whose row 0 lies in block 0.
constexpr int32_t kUnit64 = 1, kUnitWide = 2;   // ScoreUnit::shape: G = 64 (else 16), wide values
struct ScoreUnit {
    int32_t first;      // index of the first pair in `order`
    int32_t count;      // pairs
    int32_t maxN;       // max |H|
    int32_t nblocks;    // block 0 of G * RH rows, the others of G * R
    int32_t rows;       // R | RH << 8 (R: 8 or 16, and 4 for G = 64; RH: 4, 8, 12 or 16, and 1, 2, 3, 6 for G = 64)
    int32_t shape;
    int32_t block;      // strip: its block, else -1
    int32_t pad;
    int64_t rowOff;     // strips: the item's words in ScoreArgs::strips (nblocks x 64 / G x (maxN + 1))
};
// A unit without strips in 12 bytes: the list's form in the no-allocation call,
// whose scratch array holds it (40 bytes per 8 pairs of 16 lanes would refuse
// calls of 2.7 million short pairs on).
struct SlimUnit {
    int32_t first;
    uint32_t size;      // maxN | nblocks << 16
    uint32_t form;      // count | shape << 8 | rows << 16
    __host__ __device__ static SlimUnit of(const ScoreUnit &u)
    {
        return SlimUnit{u.first, (uint32_t)u.maxN | (uint32_t)u.nblocks << 16,
                        (uint32_t)u.count | (uint32_t)u.shape << 8 | (uint32_t)u.rows << 16};
    }
    __host__ __device__ ScoreUnit unit() const
    {
        return ScoreUnit{first, (int32_t)(form & 0xff), (int32_t)(size & 0xffff), (int32_t)(size >> 16), (int32_t)(form >> 16),
                         (int32_t)(form >> 8 & 0xff), -1, 0, 0};
    }
};
struct ScoreArgs {
    const uint8_t *hRes;
    const uint8_t *vRes;
    const int64_t *hOff;
    const int64_t *vOff;
    const int32_t *order;
    const ScoreUnit *units;
    const SlimUnit *slim;       // in place of `units`, or null
    int32_t nUnits;
    uint32_t *queue;            // unit counter (zeroed before the launch)
    uint64_t *rowbuf;           // slotWords (G, F) words per wave of the grid
    int64_t slotWords;
    uint64_t *strips;           // strips' bottom rows (zeroed before the launch)
    int64_t stripWords;
    uint32_t *error;            // host memory: set when a strip's wait runs past its bound
    int32_t *scores;            // indexed by pair id
    uint32_t mode;
    int32_t alpha;
    const int16_t *tTable;
    const uint32_t *dnaProfile;
    Drift drift;
};
// Waves per workgroup of a launch of `units` units: 4, or 8 with the table where
// the units fill the chip's SIMDs twice.
constexpr int kScoreTabWaves = 8;
inline int scoreWaves(bool dna, int64_t units, int numCUs) { return dna || units <= (int64_t)4 * numCUs ? 4 : kScoreTabWaves; }
hipError_t launchScore16(bool dna, int kind, const ScoreArgs &args, int gridBlocks, int waves, hipStream_t stream);
int occupancyScore16(bool dna, int kind, int waves);

// Kernel variant of the packed int16 family.
struct Variant16 {
    int G;      // lanes per pair group
    int R;      // rows per lane
    bool dna;   // v_perm profile path (alphabet <= 4)
    uint32_t track;
    bool wide = false;  // global scores: drifted values above kDriftNarrowMax
};

int wavesPerBlock16();
hipError_t launchSimple32(const Simple32Args &args, hipStream_t stream);

// One pair couple per lane (lane.hip): Variant16 with G = 1 and R in {16,
// 32}.  Work items hold up to 128 pairs with the same number of R-row
// blocks; the row buffer holds, per wave slot, laneRowCols(maxN, R) columns
// x 64 lanes of (G, F) pairs (8 bytes each).
bool laneSupported(const Variant16 &v);
int laneRowCols(int maxN, int R);
// Packed banded scores (band16.hpp): one pair couple per lane, R rows per
// block, bandUp - bandLo >= R; work items hold up to 128 pairs of one length m
// (WorkItem.count = pairs | m << 16, nblocks = (m + R) / R).  Row buffer per
// wave slot: a ring of bandRingCols(...) columns x 64 lanes x 8 bytes, in LDS
// where bandLdsRingBytes() > 0 (one ring per workgroup of `waves` waves, else
// one per wave of four).  R: 8 and 12 with LDS rings, 16 with either.
constexpr int kBandWaves = 8;
enum BandKind : int { kBandEnd = 0, kBandFree = 1, kBandLocal = 2 };   // cell (m, n); free last row / column; local
struct BandVariant {
    int R;
    bool dna;
    int kind;
    bool wide;      // values above kDriftNarrowMax
    bool lds;
    int waves;      // per workgroup
};
constexpr int bandRowCols(int maxN) { return (maxN + 3) / 4 * 4 + 5; }
int bandRingCols(int maxN, int64_t lower, int64_t upper, int R);
// LDS bytes of a workgroup's rings, 0 where they do not fit.
int bandLdsRingBytes(int bandCols);
int occupancyBand16(const BandVariant &v, int ringLdsBytes);
hipError_t launchBand16(const BandVariant &v, const FwdArgs &args, int gridBlocks, int ringLdsBytes, hipStream_t stream);
int occupancyLane16(const Variant16 &v);
hipError_t launchLane16(const Variant16 &v, const FwdArgs &args, int gridBlocks, hipStream_t stream);

// Banded global scores (banded.hip).  Pairs in `ids` passed the host's band
// checks; their band, clipped to the matrix, is lower..upper.
struct BandedArgs {
    const uint8_t *hRes;
    const uint8_t *vRes;
    const int64_t *hOff;
    const int64_t *vOff;
    const int32_t *ids;
    int32_t nIds;
    int32_t *scores;            // indexed by pair id
    int32_t gapOpen;
    int32_t gapExtend;
    uint32_t mode;              // SQMI_FREE_* bits
    int32_t alpha;
    const int32_t *table;       // alpha^2 substitution scores
    int64_t lower, upper;       // the band: lower <= j - i <= upper
    int32_t *scratch;           // wide kernel: 4 * wideStride int32 per workgroup
    int32_t wideStride;
    // Banded traceback (kBandedTrace): per ids index k, rows 1..m of S trace
    // bytes at trace + traceOff[k] (byte of cell (i, j): row i - 1, lane
    // j - i - clipped lower); per pair id the end cell and its E and F.
    uint8_t *trace;
    const int64_t *traceOff;
    int32_t *endIJ;
    int32_t *endEF;
};
// segLanes: 1..64 (power of two >= every band width: kBandedNarrow), or 0
// (kBandedWide on wideGrid workgroups).
hipError_t launchBanded(const BandedArgs &args, int segLanes, int wideGrid, hipStream_t stream);
// Forward with trace bytes for bands of at most kMaxBandTrace diagonals
// (segLanes: as in launchBanded up to 64, then a multiple of 64), then 16
// lanes per pair walk (kBandedWalk).
constexpr int kMaxBandTrace = 512;
hipError_t launchBandedTrace(const BandedArgs &args, int segLanes, hipStream_t stream);
struct BandedWalkArgs {
    const uint8_t *hRes;
    const uint8_t *vRes;
    const int64_t *hOff;
    const int64_t *vOff;
    const int32_t *ids;
    int32_t nIds;
    int32_t segLanes;
    int64_t lower;
    int64_t upper;
    const uint8_t *trace;
    const int64_t *traceOff;
    const int32_t *scores;
    const int32_t *endIJ;
    const int32_t *endEF;
    int32_t *counts;
    int32_t alpha;
    int32_t local;
    int32_t linear;
    uint8_t *ops;
    const int64_t *opOff;
    int64_t *opLen;
    int64_t *begins;
};
hipError_t launchBandedWalk(const BandedWalkArgs &args, hipStream_t stream);
// scores[ids[k]] = value for k < n.
hipError_t launchFillScores(int32_t *scores, const int32_t *ids, int n, int32_t value, hipStream_t stream);
// Rows written at the ends of their segments [off[i], off[i + 1]) of src,
// len[i] bytes each, copied back to back to dst + off[0]; start receives the
// n + 1 exclusive prefix sums of len (device memory throughout).
hipError_t launchPackRows(const uint8_t *src, const int64_t *off, const int64_t *len, int64_t *start, uint8_t *dst,
                          int64_t n, hipStream_t stream);
// p[0 .. n) = value by a kernel (no memset node, so the call can be captured in a
// HIP graph).
hipError_t launchFill32(uint32_t *p, size_t n, uint32_t value, hipStream_t stream);
inline hipError_t launchZero32(uint32_t *p, size_t n, hipStream_t stream) { return launchFill32(p, n, 0, stream); }

// The no-allocation entry point's device array (scratch.hip): its size and
// its device address on `device`, which must be the current device; the
// address is looked up once per device.
constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
hipError_t scratchAddress(int device, void **out);

// Long pairs (int32, tiled).  A pair with m rows and n columns is cut into
// row blocks of kTileRows (bottom-aligned like the packed kernels: item row
// p + i holds pair row i, p = nblocks * kTileRows - 1 - m) and column tiles of
// tileC columns (tile t holds columns t * tileC + 1 ... (t + 1) * tileC).
// Tile (b, t) needs the bottom row of tile (b - 1, t) and the right column of
// tile (b, t - 1): the forward runs one launch per tile anti-diagonal b + t,
// and keeps every tile border as a checkpoint for the traceback.
constexpr int kTileRows = 256;
struct LongPair {
    int32_t pid;
    int32_t n, m;
    int32_t nblocks, ntiles;
    int32_t p;
    int64_t rowck;      // int32 offset of the row checkpoints: nblocks x (n + 1) x (G, F)
    int64_t colck;      // int32 offset of the column checkpoints: nblocks x ntiles x kTileRows x (G, E)
    int64_t bestck;     // local scores: offset of the pair's nblocks maxima (one per row block)
};
struct TileArgs {
    const uint8_t *hRes;
    const uint8_t *vRes;
    const int64_t *hOff;
    const int64_t *vOff;
    const LongPair *pairs;
    int32_t nPairs;
    int32_t wavesPerPair;       // forward: waves per pair in the grid (4 blocks per wave)
    int32_t diag;               // forward: tile anti-diagonal b + t
    int32_t tileC;
    int32_t *ck;                // checkpoint storage
    int32_t gapOpen;
    int32_t gapExtend;
    const uint32_t *dnaProfile;
    int32_t *scores;            // per pair id
    int32_t *endEF;             // per pair id: E, F of cell (m, n)
    uint32_t mode;              // SQMI_FREE_* / SQMI_LOCAL
    int32_t *best;              // local: per row block of each pair (LongPair::bestck), the maximum G so far
    // traceback
    uint2 *trace;               // per long pair: kRoundSlots tiles x kTileRecSteps steps x 16 lanes records
    int32_t *walk;              // per long pair: walk state (kWalkStateInts ints)
    int32_t *counts;            // per pair id: alpha^2 + 2 counts
    int32_t alpha;
    uint8_t *ops;               // rows, as in WalkArgs (optional)
    const int64_t *opOff;
    int64_t *opLen;
};
constexpr int kTileSlack = 24;        // steps per tile beyond its width (skew + prefetch)
constexpr int kWalkStateInts = 8;
// Traceback window of one round: kRoundBlocks row blocks x kRoundTiles column
// tiles recomputed with trace records (tileC = kLongTileC).
constexpr int kLongTileC = 128;
constexpr int kTileRecSteps = kLongTileC + kTileSlack;
constexpr int kRoundBlocks = 8, kRoundTiles = 16, kRoundSlots = kRoundBlocks * kRoundTiles;
hipError_t launchTileFwd32(const TileArgs &args, hipStream_t stream);
hipError_t launchTileTrace32(const TileArgs &args, hipStream_t stream);
// Scores of long pairs under free end gaps or local alignment, from the
// forward's checkpoints (free last row / column) or its running maximum.
hipError_t launchLongResult(const TileArgs &args, hipStream_t stream);
hipError_t launchTileWalkInit(const TileArgs &args, hipStream_t stream);
hipError_t launchTileWalk32(const TileArgs &args, hipStream_t stream);

// Packed long pairs, global (long16.hip): couples of pairs in strips of 64 R
// rows, R = 4, 8 or 16 rows per lane, bottom-aligned (pair row i is strip row
// p + i).  `state` and `rows` count words in LongArgs::state and ::rows.
struct LongCouple {
    int32_t pid[2];     // the second -1: none
    int32_t n[2], m[2], p[2];
    int32_t maxN;       // the larger |H|
    int32_t nb;         // strips
    int32_t chunks;     // checkpoints per strip
    int32_t pad;
    int64_t rows;       // (nb - 1) x (maxN + 1) words: bottom rows
    int64_t state;      // nb x chunks x longStateWords(R) x 64 words
};
constexpr int kLongT = 128;             // steps between checkpoints
constexpr int kLongSlackV = 512;        // growth of a strip's top row before its base is raised
constexpr int kWinChunks = 14, kWinCouples = kWinChunks / 2;   // a traceback window's chunks, waves per strip of it
constexpr int kLongWalkInts = 8;
constexpr int longSteps(int maxN) { return (maxN + 64 + 3) / 4 * 4; }
constexpr int longStateWords(int R) { return 2 * R + 4; }
constexpr int longWinStrips(int R) { return 1024 / (64 * R) + 1; }
constexpr int longRecBytes(int R) { return R == 16 ? 16 : 8; }
struct LongArgs {
    const uint8_t *hRes;
    const uint8_t *vRes;
    const int64_t *hOff;
    const int64_t *vOff;
    const LongCouple *couples;
    int32_t nCouples;
    const int2 *units;          // (couple, strip), strip by strip
    int32_t nUnits;
    uint32_t *queue;            // unit counter (zeroed before the launch)
    uint64_t *rows;             // zeroed before the launch
    uint32_t *state;            // null: no checkpoints
    uint32_t *error;            // as in ScoreArgs
    int32_t target;             // a strip's base is raised to keep its top row here
    int32_t alpha;
    const uint32_t *dnaProfile;
    Drift drift;
    int32_t *scores;            // per pair id
    int32_t *endEF;             // per pair id: E, F of cell (m, n)
    // Traceback.
    void *trace;                // per pair: longWinStrips x kWinCouples x kLongT x 64 records
    int32_t *walk;              // per pair: kLongWalkInts ints
    int32_t *counts;            // per pair id: alpha^2 + 2 counts
    int32_t linear, alwaysOpen; // gap open == / > gap extend
    uint8_t *ops;               // rows, as in WalkArgs (optional)
    const int64_t *opOff;
    int64_t *opLen;
};
hipError_t launchLong16(int R, const LongArgs &args, int numCUs, hipStream_t stream);
hipError_t launchLong16WalkInit(const LongArgs &args, hipStream_t stream);
// One round: the windows' trace records, then the walks through them.
hipError_t launchLong16Round(int R, const LongArgs &args, hipStream_t stream);

// Trace family (trace16.hpp).
constexpr int kTraceRows = 256;       // rows per block of the trace kernel
constexpr int kTraceLanes = 16;
inline int traceSteps(int maxN, int lanes) { return (maxN + lanes + 3) / 4 * 4; }   // column steps per block
// Units as ScoreArgs' (kUnit64: 64 lanes per couple, else 16), 256-row blocks
// throughout, `pad` the item's index.
struct TraceArgs {
    const uint8_t *hRes;
    const uint8_t *vRes;
    const int64_t *hOff;
    const int64_t *vOff;
    const int32_t *order;
    const ScoreUnit *units;
    int32_t nUnits;
    uint32_t *queue;
    uint64_t *rowbuf;
    int64_t slotWords;
    uint64_t *strips;
    int64_t stripWords;
    uint32_t *error;
    uint32_t mode;
    int32_t alpha;
    const int16_t *tTable;
    const uint32_t *dnaProfile;
    Drift drift;
    uint4 *trace;               // 16-byte trace records (64 per step)
    int64_t traceRecs;          // steps the buffer holds
    const int64_t *traceOff;    // per item: its first step
    TraceEnd *ends;
    const int64_t *endOff;      // per item: its first candidate
};
// track: kTrackEnd (global), the bottom / right bits of free end gaps, or kTrackLocal.
hipError_t launchTrace16(bool dna, uint32_t track, const TraceArgs &args, int gridBlocks, hipStream_t stream);
int occupancyTrace16(bool dna, uint32_t track);
hipError_t launchWalk16(const WalkArgs &args, hipStream_t stream);
hipError_t launchCounts32(const Counts32Args &args, hipStream_t stream);

}  // namespace sqmi
