// lsort_dev.h -- device helpers of the bucket sorts: the key of a record, its
// bucket in a boundary table, the segment of a tile, block scans (gfx950,
// wave64).
#pragma once
#include "device.h"
#include "lsort.h"

namespace mpsg {

// FAST: the common layout (the key in the record's first words, no bit
// shift) is taken without the word selection when the key has it (the
// condition is the same for the whole kernel; used where the registers
// allow the second code path)
template <int RW, bool FAST = false>
__device__ __forceinline__ uint64_t lkey(const uint32_t (&r)[RW], const LKey& k) {
    if (FAST && k.w0 == 0 && k.sh == 0) {
        uint64_t v = r[0];
        if constexpr (RW > 1) v |= (uint64_t)r[1] << 32;
        return (v & k.mask) ^ k.xmask;
    }
    const uint32_t a = pick_word<RW>(r, k.w0), b = pick_word<RW>(r, k.w0 + 1),
                   c = pick_word<RW>(r, k.w0 + 2);
    const uint64_t lo = (uint64_t)a | ((uint64_t)b << 32);
    const uint64_t v = k.sh ? ((lo >> k.sh) | ((uint64_t)c << (64 - k.sh))) : lo;
    return (v & k.mask) ^ k.xmask;
}

__device__ __forceinline__ uint32_t bucket_of(uint64_t key, const uint64_t* __restrict__ t) {
    int lo = 0;
#pragma unroll
    for (int step = 512; step > 0; step >>= 1)
        if (lo + step <= kLBounds && t[lo + step - 1] < key) lo += step;
    return (uint32_t)lo;
}

// bucket b of table t holds one key value only
__device__ __forceinline__ bool single_bucket(const uint64_t* __restrict__ t, int b) {
    if (b == 0) return t[0] == 0;
    if (b >= kLBounds) return false;
    return t[b - 1] + 1 == t[b];
}

// segment of a tile: the last s with tile_start[s] <= tile (the whole wave
// asks for one tile; up to 64 segments are compared by one ballot instead of
// a search of dependent loads)
__device__ __forceinline__ int seg_of_tile(const SegDev& seg, int64_t tile) {
    if (seg.nseg <= 64) {
        const int lane = threadIdx.x & 63;
        const bool in = lane < seg.nseg && seg.tile_start[lane] <= tile;
        return (int)__popcll(__ballot(in)) - 1;
    }
    return upper_index<int64_t>(seg.tile_start, seg.nseg, tile);
}

// Position of sample u of m among n records (u < m <= n; u < 2^15, n < 2^32):
// somewhere in the u-th of m equal parts, by a fixed hash of u (the finaliser of
// Appleby's MurmurHash3).  Even positions meet data of a period that divides
// n / m, such as records interleaved from several sources or a grid in row
// order, always at the same phase: 2^21 records of 128 interleaved sources were
// sampled from one source, and all others fell into two buckets.
__device__ __forceinline__ uint64_t sample_pos(uint32_t u, uint32_t m, uint64_t n) {
    uint32_t h = u;
    h ^= h >> 16;
    h *= 0x85ebca6bu;
    h ^= h >> 13;
    h *= 0xc2b2ae35u;
    h ^= h >> 16;
    return ((((uint64_t)u << 16) | (h & 0xffffu)) * n >> 16) / m;
}

// exclusive scan of B values, one per thread of a B-thread block
template <int B>
__device__ __forceinline__ uint32_t scan_block(uint32_t v, uint32_t* s_tmp /*B / 64*/) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) s_tmp[wave] = x;
    __syncthreads();
    uint32_t pre = 0;
#pragma unroll
    for (int w = 0; w < B / 64; w++) pre += (w < wave) ? s_tmp[w] : 0u;
    __syncthreads();
    return pre + x - v;
}

}  // namespace mpsg
