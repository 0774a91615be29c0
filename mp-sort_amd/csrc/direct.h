// direct.h -- the whole sort without per-rank local sorts (direct.hip).
//
// The output of the histogram sort is the stable order of all records, and
// its counts (splitters, CLT/CLE, layout) follow from that order and from
// where each rank's records went.  For up to 64 ranks the records are
// therefore partitioned once into key buckets over all ranks together and
// each bucket sorted in LDS; the counts are taken afterwards.
#pragma once
#include "lsort.h"

namespace mpsg {

constexpr int kDirectMaxP = 64;         // ranks: one lane each
constexpr int kSmallRecords = 8192;     // sorted by one launch
constexpr int kRankRecords = 4096;      // of those, by counting every record's rank
constexpr int kDirectChunk = 1024;      // sample keys sorted by one workgroup
constexpr int kDirectMaxChunks = 16;    // sample chunks

// the host tables of one call, passed by value (no upload)
struct DirectShape {
    int P;
    int W;            // buckets (2 .. kLBins)
    int S;            // sample keys (a multiple of kDirectChunk; 0: no sample)
    int tile;         // records per tile
    int64_t n;
    int64_t ntiles;   // tiles never cross a rank
    int64_t begin[kDirectMaxP + 1];
    int64_t tile_start[kDirectMaxP + 1];
    int64_t C[kDirectMaxP + 1];
};

// device arrays of one call
struct DirectWork {
    int64_t *C, *begin, *count, *tile_start;  // tables copied from the shape
    uint64_t* chunks;     // S sample keys, each chunk sorted
    uint64_t* raw;        // kLBins: the sample keys at the boundaries
    uint64_t* tables;     // kLBins: the boundaries (kLBounds used)
    uint32_t* tot;        // kLBins: records per bucket
    int64_t* base;        // kLBins: first output record of every bucket
    uint16_t* tile_cnt;   // ntiles * kLBins
    uint32_t* tile_off;   // ntiles * kLBins: offset of the tile's run in its bucket
    uint16_t* bkt;        // n: bucket of every record
    uint32_t* lists;      // 8: [0] oversized, [1] LDS radix, [2] 1024-thread form, [7] counting blocks done
    uint32_t *hard, *medium;  // kLBins each
    int64_t* overflow;    // 2 * kLBins
    uint32_t* err;        // 4: [0] layout and splitter flags, [1] scatter flags
    long long* checksum;  // [0] in, [1] out
    int64_t *myclt, *mycle, *myC, *send;
    uint64_t* cross;      // kDirectMaxP^2: CLE << 32 | CLT by splitter and rank, for the layout
    uint64_t *split, *pminmax;
    const uint64_t* prop;     // a model's proposals for the splitters (may be null)
    unsigned long long* acc;  // 4, zero between calls: a small sort's blocks done and sums
};

// what the host reads at the end, written to pinned memory by the last kernel
struct DirectResult {
    uint32_t err, scatter_err;
    uint32_t lists[4];    // [3]: digit passes of the one-workgroup sort
    long long sums[2];
    uint32_t buckets;     // fine buckets of the two-level form
    uint32_t exact;       // splitters that the model proposed
};

// start / stop (here and below, may be null): events of the launch itself
// sample and its sort (two launches, one up to kDirectChunk keys); also writes
// the tables of the shape and clears the counters (the checksums too when
// clear_sums)
int launch_direct_sample(int rw, const void* src, const LKey& lk, const DirectShape& sh, const DirectWork& w,
                         bool clear_sums, hipEvent_t start, hipStream_t st);
// bucket of every record, counts per tile, and the tiles' offsets
int launch_direct_count(int rw, const void* src, const LKey& lk, const DirectShape& sh, const DirectWork& w,
                        long long* checksum, hipStream_t st);
// splitters, counts and layout from the sorted records out and the
// partitioned ones part (whose single-value buckets are not read), and the
// call's results into res (pinned host memory)
int launch_direct_counts(int rw, const void* out, const void* part, const LKey& lk, const DirectShape& sh,
                         const DirectWork& w, DirectResult* res, hipEvent_t stop, hipStream_t st);

// at most kSmallRecords records sorted by one launch, with the splitters,
// counts and layout (w: C, myclt, mycle, myC, send, split, pminmax, cross,
// acc).  rw = 0: records of elsize bytes with key_bytes key bytes at key_off.
// apart: in and out do not overlap (otherwise they are the same)
int launch_small_sort(int rw, const void* src, void* dst, const LKey& lk, int elsize, int key_off, int key_bytes,
                      const DirectShape& sh, const DirectWork& w, bool checksum, bool apart, DirectResult* res,
                      hipEvent_t start, hipEvent_t stop, hipStream_t st);

}  // namespace mpsg
