// wide.h -- the sort of up to 64 ranks in two partition levels (wide.hip), for
// sizes that one partition into in-LDS buckets does not reach.
//
// Every tile of 6144 records is grouped by bucket in its own place, so no
// counting pass over the records comes first and every write is contiguous;
// the next level gathers a bucket's runs from the tiles in tile order, which
// keeps the sort stable.  Level 1 groups the input by up to 512 coarse buckets
// (boundaries from a sample of all records), level 2 the records of every
// coarse bucket by up to 512 fine ones (from a sample of that bucket), and
// groups of neighbouring fine buckets are gathered and sorted in LDS.
#pragma once
#include "direct.h"

namespace mpsg {

constexpr int kWideBuckets = 512;                // buckets of one level, at most
constexpr int kWideTile = 6144;                  // records per tile
constexpr int kWideStride = kWideBuckets + 8;    // run starts of a tile
constexpr int kWideRuns = 256;                   // tiles of a coarse bucket, at most
constexpr int kWideSamples = 4096;               // sample keys of a coarse bucket
constexpr int kWideCopy = 4096;                  // records of one copy task
constexpr int kWideCap = kMergeCap;              // a group of fine buckets sorted by 512 x 6 threads and records
constexpr int kWideFine = 1024;                  // records per fine bucket while 512 buckets suffice
// The largest call: an average coarse bucket of 7/16 of what kWideRuns tiles
// hold.  Its boundaries are 32 sample keys apart, so bucket sizes deviate by 18%
// on average: one call in 100,000 of randomly ordered keys has a bucket above
// the limit and takes the per-rank form after all, at 400 M records one in 700,
// at 2^29 nineteen in twenty.
constexpr int64_t kWideMaxRecords = (int64_t)kWideBuckets * kWideRuns * kWideTile / 16 * 7;

// a group of neighbouring fine buckets [f, fe) and its tiles' runs
struct WideBucket {
    uint32_t tile0;    // first tile of its coarse bucket
    uint32_t first;    // first record of that tile
    uint16_t ntiles, f, fe, pad;
};

struct WideWork {
    int W, avg;                // coarse buckets; records per fine bucket
    int64_t n, nt, ntpad;      // records, level 1 tiles, entries of a row of off and loc
    int64_t nt2, nfine;        // level 2 tiles and fine buckets, at most
    int64_t ngrid;             // groups sorted by one workgroup each (wide_grid); those past it are listed
    uint32_t cap;              // largest group sorted in LDS (kChunkCap, less by the capacity fault hook)
    const uint64_t* raw;       // W - 1 sample keys at the coarse boundaries
    uint64_t* tables;          // kWideBuckets coarse boundaries
    uint64_t* tables2;         // W rows of kWideBuckets fine boundaries
    uint32_t* tile_beg;        // nt: first record of every level 1 tile
    uint16_t *ex1, *ex2;       // nt / nt2 rows of kWideStride: start of every bucket's run in its tile
    uint32_t* part;            // rows of kWideBuckets: coarse counts of 64 tiles, then their prefix
    uint32_t* off;             // W rows of ntpad: the coarse bucket's records in earlier tiles
    uint16_t* loc;             // W rows of ntpad: its run's start in the tile
    uint32_t* tot;             // kWideBuckets: records per coarse bucket
    uint32_t *cbase, *ctile, *cfine;  // kWideBuckets + 1: first record, level 2 tile, fine bucket
    uint32_t* cw;              // kWideBuckets: fine buckets (0: one key value, or empty)
    uint32_t* first;           // nt2: level 1 tile of the level 2 tile's first record
    WideBucket* desc;          // nfine (groups, at most one per fine bucket)
    uint32_t* fcnt;            // nfine: records of the group
    int64_t* fbase;            // nfine: its first output record
    uint32_t *medium, *hard;   // nfine each
    uint2* copy;               // {group, first record}, ncopy at most
    int64_t ncopy;
    int64_t* overflow;         // {base, count} of the groups above the in-LDS capacity
    int max_overflow;
    uint32_t* lists;           // 8: [0] oversized, [1] LDS radix, [2] 1024-thread form, [4] copy tasks,
                               // [5] set: a coarse bucket of several values has too many tiles, [6] groups
    const uint32_t* tile_c;    // segments: coarse bucket (segment) of every level 2 tile
    uint32_t* tally;           // 2 * kDirectMaxP^2: records below and at most each splitter, by rank
};

// level 1 of [0, n) (ranks: sd): src -> dst tile by tile, the coarse counts
// and offsets, and the coarse buckets' samples.  clears tally; lists are zero
// before (launch_direct_sample)
int launch_wide_level1(int rw, const void* src, void* dst, const LKey& lk, const SegDev& sd, const WideWork& w,
                       long long* checksum, hipStream_t st);
// fine boundaries and level 2: src (level 1's dst) -> dst tile by tile, the
// coarse buckets of one key value straight to out; then the groups of fine
// buckets
int launch_wide_level2(int rw, const void* src, void* dst, void* out, const LKey& lk, const WideWork& w,
                       long long* checksum_out, hipStream_t st);
// every group gathered from recs and sorted into out, those above 3072
// records by larger workgroups and crowded ones by the LDS radix sort; buckets
// above 9216 records are copied to their places (those of several values,
// listed in overflow, for the radix path)
int launch_wide_sort(int rw, const void* recs, void* out, const LKey& lk, const WideWork& w, long long* checksum_out,
                     hipStream_t st);
// the listed oversized buckets of several values, in place in out, by digit
// passes through the same positions of tmp
int launch_wide_big(int rw, void* out, void* tmp, const LKey& lk, const WideWork& w, hipStream_t st);
// independent segments (w.W of them, each at most kWideSegMax records, as
// coarse buckets whose tot, cbase, ctile, cw and tile_c the caller has
// set): src -> out through tmp (src may equal out); nothing but kernels
// (512 buckets of 1843 records on average: 1.9 deviations of a size estimated
// from 8 sample keys below 3072, 4.2 below the 4608 of the listed form)
constexpr int64_t kWideSegMax = (int64_t)kWideBuckets * 1843;
// groups of n records in W coarse buckets: two neighbours hold more than
// 3072 records together unless one of them stands alone
inline int64_t wide_grid(int64_t n, int64_t W) { return (n / (kWideCap / 2) + 2 * W + 7) / 8 * 8; }
int launch_wide_segments(int rw, const void* src, void* tmp, void* out, const LKey& lk, const WideWork& w,
                         hipStream_t st);
// splitters, counts and layout (as launch_direct_counts): part is level 1's dst
int launch_wide_counts(int rw, const void* out, const void* part, const LKey& lk, const DirectShape& sh,
                       const DirectWork& d, const WideWork& w, DirectResult* res, hipEvent_t stop, hipStream_t st);

}  // namespace mpsg
