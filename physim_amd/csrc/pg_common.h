// Shared host/device definitions of the physim_gpu engine.
#pragma once

#include <stdint.h>

#include "physim_gpu.h"

namespace pg {

constexpr int kBlock = 256;        // threads per block (4 wave64)
constexpr int kSortTile = 2048;    // keys per radix-sort tile
constexpr int kSortThreads = 512;  // threads per radix-sort tile
constexpr int kSortItems = kSortTile / kSortThreads;  // keys per thread
constexpr int kScanItems = 4;      // counts per thread in the node-offset scan
constexpr int kScanTile = kBlock * kScanItems;
constexpr int kMaxPasses = 8;      // 8-bit digits over a 64-bit key
constexpr int kKeyThreads = 512;   // threads of a key-building block (one sort tile)
constexpr int kBucketKeys = 1664;  // keys per bucket of the sample sort (on average; steady-state
                                   // buckets stay within 2048, the slot sort's reach)
// The same in small batches, which are far from filling the GPU: shorter
// buckets are one or two keys a thread, and more blocks (mean 1664: sort of
// 10,002 bodies 12.1 us, 131,072 14.4, 524,288 16.4; 384: 9.0 and 9.9, but 18 at
// 524,288, where past kMaxBuckets splitters keys take longer too; 1024: 15.1).
constexpr int kBucketKeysFew = 384;    // up to kFewBodies bodies
constexpr int kBucketKeysMore = 1024;  // up to kMoreBodies
constexpr uint64_t kFewBodies = 1u << 17, kMoreBodies = 1u << 19;
constexpr uint64_t kFewKeys = 1u << 18;  // up to here a thread builds one key, not two
constexpr int kGatherKeys = 16384;  // batches whose sort blocks collect their own keys (no scatter)
constexpr int kBucketCap = 4096;   // largest bucket sorted in LDS (larger ones: in HBM)
constexpr int kMinBucketKeys = 256;  // smallest mean bucket a tuning may ask for
constexpr int kBucketThreads = 512;   // threads of a bucket-sorting block (up to 8 keys each)
constexpr int kMaxBuckets = 1024;  // buckets whose splitters every key tile holds in LDS
constexpr int kMaxWideBuckets = 8192;  // more buckets: splitters in HBM behind a coarse table
constexpr int kWideGroup = 8;      // splitters per coarse-table entry (kMaxWideBuckets / kWideGroup
                                   // entries fit a tile's LDS)
constexpr int kSampleOver = 4;     // splitter samples per bucket (sampling from unsorted keys)
constexpr int kWideSampleOver = 2; // the same with more than kMaxBuckets buckets (128 KB of LDS)
constexpr int kSplitThreads = 1024;  // threads of the splitter block
constexpr int kQuantiles = 256;    // per bucket: quantiles of the previous sorted keys
constexpr int kScanThreads = 1024;  // threads of a per-digit scan over the sort tiles
constexpr int kExtentChunk = 4096; // bodies per extent partial
constexpr uint32_t kExtentBlocks = 256;  // blocks of the extent pass (each takes chunks in turn)
constexpr int kNodeTile = 1024;    // sorted bodies per node-building block
constexpr int kNodeThreads = 512;  // threads per node-building block (two bodies each)
constexpr int kNodeLds = 2016;     // kNodeTile bodies + up to kNodeLds - kNodeTile internal nodes: built one
                                   // node per thread (more internal nodes: body by body). Uniform
                                   // quadtrees have 0.7 per body, up to 0.9 in a tile: with a list of
                                   // 768 a build of 50,003 bodies took 34 us, with 992 (the most at
                                   // three blocks a CU) 21
constexpr int kFewTiles = 64;      // batches of at most this many node tiles: no scan over the tiles apart
constexpr int kTopSlots = 65;      // tree levels 0..64: one tile-spanning node each
constexpr int kMaxTieRun = 256;    // longest run of equal keys ordered by their deep keys
constexpr int kMaxLcp = 64;        // deepest common prefix, in levels, of two bodies: the
                                   // reference recurses to depth 64 (octree.rs:60-62)
constexpr int kDirectUnit = 32;    // sources per group of the FP64 direct sum: a multiple of this
// A line of the direct sum's partial sums: those of a target tile's bodies over
// one source tile (mixed precision, FP32), or half of those over one group (FP64
// words, two lines). A target tile's lines lie together, the tiles in batch order.
constexpr int kPartFloats = 3 * kBlock;
constexpr uint64_t kPartLine = kPartFloats * sizeof(float);
constexpr int kDeepWords = 3;      // words of a tied body's deep key
static_assert(kMaxLcp + 1 == kTopSlots, "every level of an internal node has its slot");

// Deep key of a body whose first key word ties with a neighbour's: the
// digits of the levels past the first word, from the same descent.
struct DeepKey {
    uint64_t w[kDeepWords];
};
constexpr int kComSpanGroups = 5;   // level groups (of 4 waves) per tile in k_com_span
static_assert(kScanTile == kNodeTile, "node offsets and node building share their tiles");
static_assert(kNodeTile == 2 * kNodeThreads, "the partial sums take two bodies per thread");
static_assert(kTopSlots <= kBlock, "per-level tables are filled by one thread per level");
static_assert(kSortTile % kKeyThreads == 0 && kKeyThreads >= 256, "whole key tiles, a digit per thread");
static_assert(kSortTile % kSortThreads == 0 && kSortThreads >= 256, "whole sort tiles, a digit per thread");

// Device-side error bits (sticky per segment), mapped to pg_status on the host.
enum : uint32_t {
    kErrDepth = 1u << 0,
    kErrCoincident = 1u << 1,
    kErrNonFinite = 1u << 2,
    kErrCapacity = 1u << 3,
};

struct SegState;

// A body's tag, the fourth word of its previous-position record: its upload
// index (low 32 bits) and its fixed flag (bit 32), a bit pattern that no
// arithmetic touches.
__host__ __device__ inline double make_tag(uint32_t id, bool fixed) {
    return __builtin_bit_cast(double, (uint64_t)id | ((uint64_t)(fixed ? 1u : 0u) << 32));
}
__host__ __device__ inline uint32_t tag_id(double t) {
    return (uint32_t)__builtin_bit_cast(uint64_t, t);
}
__host__ __device__ inline bool tag_fixed(double t) {
    return (__builtin_bit_cast(uint64_t, t) >> 32) != 0;
}

// One simulation's view inside a batched launch: the current state (src) and
// the buffer the step writes (dst), both SoA in the order of the previous
// build's Morton sort.
struct SegDesc {
    // per body: (x, y, z, m) and (x_prev, y_prev, z_prev, tag); velocities
    const double4* spos; const double4* sprv;
    const double* svx; const double* svy; const double* svz;
    double4* dpos; double4* dprv;
    double* dvx; double* dvy; double* dvz;
    uint64_t off;   // first global (batch) index of this segment
    uint64_t n;
    double theta, e, dt;
    uint32_t seg;
    uint32_t count; // per-body interaction counts into counts[] and step statistics
    int64_t* counts;
    struct SegState* st;
    uint32_t chunk0;  // first extent chunk of this segment
    uint32_t nchunks;
    uint32_t tile0;   // first node tile of this segment (node tiles start at its first body)
    uint32_t nsplit;  // direct sum, mixed precision: ranges of source tiles summed apart
    uint32_t ngroup;  // direct sum: blocks summing one target tile, each over a group of source tiles
    uint32_t fine;    // mixed precision: more groups than ranges (every tile's partial sum is kept)
    uint64_t part_line;  // direct sum with ngroup > 1: the segment's first line of partial sums
    double near;      // near field in widths of the body's own leaf cell (0: off)
};

// Per-segment device scalars.
struct SegState {
    uint64_t extent_bits;   // max |coord| as the bit pattern of a non-negative double
    uint64_t interactions;
    uint64_t steps_done;
    uint32_t history;       // 1 when the Stormer history is valid for this step
    uint32_t err;
    uint32_t max_level;
    uint32_t vperm;         // velocities must travel with the state (not yet derivable)
};

// Internal tree node record, one 64-byte line: what the walk's opening test
// reads in the first half (fetched through the scalar unit), the source a body
// that takes the node adds in the second (the form of a leaf's position
// record). Skip and level are kept as the walk uses them: a byte offset into
// the span array (8 bytes per node; times 8, into the records) and the
// exponent of 4^level.
struct NodeHot {
    double cx, cy, cz;      // geometric centre (reference rounding)
    uint32_t skip8;         // 8 * index of the next internal node after this subtree
    uint32_t level2;        // 2 * level
    double mx, my, mz;      // centre of mass
    double mass;
};

// Batch-wide counters reset at the start of every step.
struct StepCounters {
    uint32_t gen;           // bumped per step: versions tile-spanning node slots
    uint32_t top_levels;    // 1 + deepest level of a tile-spanning node (0: none)
    uint64_t sort_tag;      // batch whose sorted keys the sample sort left (0: none)
    uint64_t ext_tag;       // batch whose current positions the extent partials hold (0: none)
    uint32_t split_prev;    // this step's splitters may come from those keys
    uint32_t quantiles;     // they did: finer quantiles per bucket were taken too
};

}  // namespace pg
