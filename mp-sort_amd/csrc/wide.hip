// wide.hip -- the sort of up to 64 ranks in two partition levels (see wide.h).
// Its output is the stable order that the reference's FirstSort, exchange and
// SecondSort (mpsort-mpi.c:369,571-597) produce; the splitters and counts of
// the histogram sort (mpsort-mpi.c:375-510) are read off the result.
#include <hip/hip_ext.h>

#include "layout_dev.h"
#include "lsort_dev.h"
#include "wide.h"

namespace mpsg {

constexpr int kWBlock = 512, kWWaves = kWBlock / 64, kWItems = kWideTile / kWBlock;
constexpr int kWSpan = 64 * kWItems;  // records of a wave
static_assert(kWBlock == kWideBuckets, "a thread per bucket");

// boundary e of a table made from raw sample keys (nb of them): where
// boundaries repeat a key v, the first becomes v - 1, so that (v - 1, v]
// holds that key alone
__device__ __forceinline__ uint64_t wide_boundary(const uint64_t* raw, int e, int nb) {
    if (e >= nb) return ~0ull;
    const uint64_t v = raw[e];
    const bool first = e == 0 || raw[e - 1] < v;
    const bool repeated = e + 1 < nb && raw[e + 1] == v;
    return first && repeated && v > 0 ? v - 1 : v;
}
// bucket b of a table of nb boundaries holds one key value only
__device__ __forceinline__ bool wide_single(const uint64_t* t, int b, int nb) {
    if (b >= nb) return false;
    return b == 0 ? t[0] == 0 : t[b - 1] + 1 == t[b];
}

// LDS of a level 2 tile while its records are located: the runs (a run's
// position in src less its position in the tile), a bit per run start, and
// the runs before every word of those bits
struct WideRunTab {
    uint32_t run[kWideTile];
    uint32_t bits[kWideTile / 32];
    uint32_t pref[kWideTile / 32];
    __device__ __forceinline__ uint32_t at(uint32_t q) const {
        const uint32_t i = pref[q >> 5] + __popc(bits[q >> 5] & (0xffffffffu >> (31u - (q & 31u)))) - 1u;
        return run[i] + q;
    }
};

// Coarse bucket of level 2 tile t: the tiles' prefix is compared by a thread
// per bucket.  s_tmp: kWWaves words.
__device__ __forceinline__ int wide_coarse_of(const WideWork& w, uint32_t t, uint32_t* s_tmp) {
    const int tid = threadIdx.x;
    const uint64_t m = __ballot(tid < w.W && w.ctile[tid + 1] <= t);
    if ((tid & 63) == 0) s_tmp[tid >> 6] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t c = 0;
#pragma unroll
    for (int q = 0; q < kWWaves; q++) c += s_tmp[q];
    __syncthreads();
    return (int)c;
}

// The runs of records [p0, p1) of coarse bucket c (level 2 tile `tile`) in
// level 1's tiles, a thread per level 1 tile.  s_w: 2 (kWWaves + 1) words.
__device__ __forceinline__ void wide_locate(const WideWork& w, int c, uint32_t tile, uint32_t p0, uint32_t p1,
                                            WideRunTab& rt, uint32_t* s_w) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if (tid < kWideTile / 32) rt.bits[tid] = 0;
    const uint32_t s0 = w.first[tile];
    const uint32_t s1 = tile + 1 < w.ctile[c + 1] ? w.first[tile + 1] + 1 : (uint32_t)w.nt;
    const uint32_t* off = w.off + (int64_t)c * w.ntpad;
    const uint16_t* loc = w.loc + (int64_t)c * w.ntpad;
    const uint64_t lt = __lanemask_lt();
    __syncthreads();
    uint32_t runs = 0;
    int par = 0;
    for (uint32_t sb = s0; sb < s1; sb += kWBlock, par ^= 1) {
        const uint32_t s = sb + tid;
        const bool in = s < s1;
        const uint32_t o = in ? off[s] : p1, e = in ? off[s + 1] : p1;
        const uint32_t from = in ? w.tile_beg[s] + loc[s] : 0u;
        const uint32_t a = max(o, p0), z = min(e, p1);
        const bool has = in && a < z;
        const uint64_t m = __ballot(has);
        uint32_t* sw = s_w + par * (kWWaves + 1);
        if (lane == 0) sw[wave] = (uint32_t)__popcll(m);
        if (tid == kWBlock - 1) sw[kWWaves] = e;
        __syncthreads();
        uint32_t idx = runs + (uint32_t)__popcll(m & lt);
#pragma unroll
        for (int q = 0; q < kWWaves; q++) {
            idx += q < wave ? sw[q] : 0u;
            runs += sw[q];
        }
        if (has) {
            const uint32_t q = a - p0;
            atomicOr(&rt.bits[q >> 5], 1u << (q & 31u));
            rt.run[idx] = from + (a - o) - q;
        }
        if (sw[kWWaves] >= p1) break;
    }
    __syncthreads();
    const uint32_t cnt = tid < kWideTile / 32 ? (uint32_t)__popc(rt.bits[tid]) : 0u;
    const uint32_t ex = scan_block<kWBlock>(cnt, s_w);
    if (tid < kWideTile / 32) rt.pref[tid] = ex;
    __syncthreads();
}

// ---------------------------------------------------------------------------
// One tile grouped by bucket, stably, and written to its own place: records
// loaded wave-major (12 loads of a thread in flight), their buckets searched
// in LDS, ranked by ballots among the lanes of a wave and by counters across
// its items and the waves, and staged through LDS 8 bytes of a record at a
// time so that two workgroups share a CU.  kLevel1 reads the input in place;
// kLevel2 reads the runs of its coarse bucket; kSegment is level 2 of a
// segment, which lies in one piece.
// 12 records per thread: with 16 (tiles of 8192) the registers spilled, and
// the two levels of 2^28 x 16 B took 3.00 and 3.35 ms instead of 2.11 and 2.30
// (8.6 GB each: 4.1 and 3.7 TB/s; level 2 2.45 ms, 3.5 TB/s, since a coarse
// bucket of that size has 512 fine ones instead of 285).
enum { kLevel1, kLevel2, kSegment };
template <int RW, int MODE>
__global__ __launch_bounds__(kWBlock, 4) void wide_part_kernel(const uint32_t* __restrict__ src,
                                                               uint32_t* __restrict__ dst, uint32_t* __restrict__ out,
                                                               LKey lk, SegDev seg, WideWork w,
                                                               long long* __restrict__ checksum) {
    constexpr int G = 4;  // records whose searches advance together
    union Stage {
        uint2 rec[kWideTile];
        WideRunTab rt;
    };
    __shared__ __attribute__((aligned(16))) Stage s;
    __shared__ uint16_t s_whist[kWWaves][kWideBuckets];
    __shared__ uint64_t s_tab[kWideBuckets];
    __shared__ uint32_t s_excl[kWideBuckets];
    __shared__ uint32_t s_tmp[2 * (kWWaves + 1)];
    __shared__ long long s_sum[kWWaves];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const uint32_t tile = blockIdx.x;
    uint32_t begin;  // first record of the tile in dst
    int cnt, nw;
    uint16_t* ex;
    if constexpr (MODE != kLevel1) {
        if (w.lists[5] || tile >= w.ctile[w.W]) return;
        const int c = MODE == kSegment ? (int)w.tile_c[tile] : wide_coarse_of(w, tile, s_tmp);
        const uint32_t p0 = (tile - w.ctile[c]) * (uint32_t)kWideTile, n = w.tot[c];
        begin = w.cbase[c] + p0;
        cnt = (int)min((uint32_t)kWideTile, n - p0);
        nw = (int)w.cw[c];
        ex = w.ex2 + (int64_t)tile * kWideStride;
        s_tab[tid] = tid < nw - 1 ? w.tables2[(int64_t)c * kWideBuckets + tid] : ~0ull;
        if constexpr (MODE == kLevel2) wide_locate(w, c, tile, p0, p0 + (uint32_t)cnt, s.rt, s_tmp);
    } else {
        const int j = seg_of_tile(seg, tile);
        begin = (uint32_t)(seg.begin[j] + (int64_t)(tile - (uint32_t)seg.tile_start[j]) * kWideTile);
        cnt = (int)min((int64_t)kWideTile, seg.begin[j] + seg.count[j] - (int64_t)begin);
        nw = w.W;
        ex = w.ex1 + (int64_t)tile * kWideStride;
        const uint64_t t = wide_boundary(w.raw, tid, nw - 1);
        s_tab[tid] = t;
        if (tile == 0) w.tables[tid] = t;
        if (tid == 0) w.tile_beg[tile] = begin;
    }
    uint32_t r[kWItems][RW];
#pragma unroll
    for (int k = 0; k < kWItems; k++) {
        const uint32_t q = (uint32_t)min(wave * kWSpan + k * 64 + lane, cnt - 1);
        RecIO<RW>::load(src, (int64_t)(MODE == kLevel2 ? s.rt.at(q) : begin + q), r[k]);
    }
    if (MODE == kLevel1 || (MODE == kLevel2 && nw == 0)) {
        // level 1 sums the input; a coarse bucket of one key value is in its
        // final order, and summed as output
        if (checksum) {
            long long cs = 0;
#pragma unroll
            for (int k = 0; k < kWItems; k++) {
                int one = 0;
#pragma unroll
                for (int q = 0; q < RW; q++) one += sbyte_sum(r[k][q]);
                cs += wave * kWSpan + k * 64 + lane < cnt ? one : 0;
            }
            cs = wave_sum_ll(cs);
            if (lane == 0) s_sum[wave] = cs;
            __syncthreads();
            if (tid == 0) {
                for (int q = 1; q < kWWaves; q++) cs += s_sum[q];
                atomicAdd((unsigned long long*)checksum, (unsigned long long)cs);
            }
        }
        if (nw == 0) {
#pragma unroll
            for (int k = 0; k < kWItems; k++) {
                const int q = wave * kWSpan + k * 64 + lane;
                if (q < cnt) RecIO<RW>::store(out, (int64_t)begin + q, r[k]);
            }
            return;
        }
    }
    for (int i = tid; i < kWWaves * kWideBuckets / 2; i += kWBlock) reinterpret_cast<uint32_t*>(&s_whist[0][0])[i] = 0;
    __syncthreads();  // the table and the cleared counters; every run is located
    int step0 = 0, nbits = 0;
    if (nw > 1) {
        nbits = 32 - __clz(nw - 1);
        step0 = 1 << (nbits - 1);
    }
    uint32_t dl[kWItems];  // bucket, then | rank in the wave << 16, then the staged position
#pragma unroll
    for (int h = 0; h < kWItems / G; h++) {
        uint64_t key[G];
        int lo[G];
#pragma unroll
        for (int k = 0; k < G; k++) {
            key[k] = lkey<RW, true>(r[h * G + k], lk);
            lo[k] = 0;
        }
        for (int step = step0; step > 0; step >>= 1) {
            uint64_t v[G];
#pragma unroll
            for (int k = 0; k < G; k++) v[k] = s_tab[lo[k] + step - 1];
#pragma unroll
            for (int k = 0; k < G; k++) lo[k] += v[k] < key[k] ? step : 0;
        }
#pragma unroll
        for (int k = 0; k < G; k++) dl[h * G + k] = (uint32_t)lo[k];
    }
    volatile uint16_t* wh = s_whist[wave];
    const uint64_t lt_mask = __lanemask_lt();
#pragma unroll
    for (int k = 0; k < kWItems; k++) {
        const bool valid = wave * kWSpan + k * 64 + lane < cnt;
        const uint32_t d = dl[k];
        uint64_t peers = __ballot(valid);
        for (int b = 0; b < nbits; b++) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            peers &= bit ? bb : ~bb;
        }
        const uint32_t rank = __popcll(peers & lt_mask);
        const uint32_t base = wh[d];  // (lanes past the tile's end rank nothing)
        dl[k] = d | ((base + rank) << 16);
        if (valid && rank == 0) wh[d] = (uint16_t)(base + __popcll(peers));
    }
    __syncthreads();
    {
        uint32_t acc = 0;
#pragma unroll
        for (int q = 0; q < kWWaves; q++) {
            const uint32_t c = s_whist[q][tid];
            s_whist[q][tid] = (uint16_t)acc;
            acc += c;
        }
        const uint32_t e = scan_block<kWBlock>(acc, s_tmp);
        s_excl[tid] = e;
        if (tid <= nw) ex[tid] = (uint16_t)e;
        if (tid == 0 && nw == kWideBuckets) ex[kWideBuckets] = (uint16_t)cnt;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kWItems; k++) {
        const uint32_t d = dl[k] & 0xffffu;
        dl[k] = s_excl[d] + s_whist[wave][d] + (dl[k] >> 16);
    }
#pragma unroll
    for (int ph = 0; ph < RW / 2; ph++) {
        if (ph) __syncthreads();
#pragma unroll
        for (int k = 0; k < kWItems; k++)
            if (wave * kWSpan + k * 64 + lane < cnt) s.rec[dl[k]] = make_uint2(r[k][2 * ph], r[k][2 * ph + 1]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kWItems; k++) {
            const uint2 v = s.rec[k * kWBlock + tid];
            r[k][2 * ph] = v.x;
            r[k][2 * ph + 1] = v.y;
        }
    }
#pragma unroll
    for (int k = 0; k < kWItems; k++) {
        const int i = k * kWBlock + tid;
        if (i < cnt) RecIO<RW>::store(dst, (int64_t)begin + i, r[k]);
    }
}

// ---------------------------------------------------------------------------
// Coarse counts: part[k][c] = records of bucket c in tiles 64 k .. 64 k + 63,
// made a prefix over k by wide_scan_kernel.
__global__ __launch_bounds__(kWideBuckets) void wide_sums_kernel(WideWork w) {
    const int c = threadIdx.x;
    if (c >= w.W) return;
    const int64_t t0 = (int64_t)blockIdx.x * 64;
    constexpr int U = 16;
    uint32_t sum = 0;
    for (int q0 = 0; q0 < 64; q0 += U) {
        uint32_t a[U], b[U];
#pragma unroll
        for (int q = 0; q < U; q++) {
            const int64_t t = min(t0 + q0 + q, w.nt - 1);
            a[q] = w.ex1[t * kWideStride + c];
            b[q] = w.ex1[t * kWideStride + c + 1];
        }
#pragma unroll
        for (int q = 0; q < U; q++) sum += t0 + q0 + q < w.nt ? b[q] - a[q] : 0u;
    }
    w.part[(int64_t)blockIdx.x * kWideBuckets + c] = sum;
}

// a block per 64 buckets, its 16 waves over equal runs of rows
__global__ __launch_bounds__(1024) void wide_scan_kernel(WideWork w, int64_t rows) {
    __shared__ uint32_t s_part[16][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int b = blockIdx.x * 64 + lane;
    const int64_t per = (rows + 15) / 16;
    const int64_t t0 = min(rows, wave * per), t1 = min(rows, t0 + per);
    constexpr int U = 16;
    uint32_t sum = 0;
    for (int64_t t = t0; t < t1; t += U) {
        uint32_t c[U];
#pragma unroll
        for (int q = 0; q < U; q++) c[q] = t + q < t1 ? w.part[(t + q) * kWideBuckets + b] : 0u;
#pragma unroll
        for (int q = 0; q < U; q++) sum += c[q];
    }
    s_part[wave][lane] = sum;
    __syncthreads();
    uint32_t run = 0, all = 0;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const uint32_t c = s_part[q][lane];
        run += q < wave ? c : 0u;
        all += c;
    }
    if (wave == 0) w.tot[b] = b < w.W ? all : 0u;
    for (int64_t t = t0; t < t1; t += U) {
        uint32_t c[U];
#pragma unroll
        for (int q = 0; q < U; q++) c[q] = t + q < t1 ? w.part[(t + q) * kWideBuckets + b] : 0u;
#pragma unroll
        for (int q = 0; q < U; q++) {
            if (t + q < t1) w.part[(t + q) * kWideBuckets + b] = run;
            run += c[q];
        }
    }
}

// the coarse buckets' places, level 2 tiles and fine buckets; clears the
// splitter tallies
__global__ __launch_bounds__(kWideBuckets) void wide_plan_kernel(WideWork w) {
    __shared__ uint32_t s_tmp[kWWaves];
    const int c = threadIdx.x;
    const uint32_t n = c < w.W ? w.tot[c] : 0u;
    const uint32_t tiles = (n + kWideTile - 1) / kWideTile;
    uint32_t nf = 0;
    if (n > 0 && !wide_single(w.tables, c, w.W - 1)) {
        nf = min((uint32_t)kWideBuckets, (n + w.avg - 1) / (uint32_t)w.avg);
        if (tiles > (uint32_t)kWideRuns) w.lists[5] = 1;
    }
    const uint32_t b = scan_block<kWideBuckets>(n, s_tmp);
    const uint32_t t = scan_block<kWideBuckets>(tiles, s_tmp);
    const uint32_t f = scan_block<kWideBuckets>(nf, s_tmp);
    w.cbase[c] = b;
    w.ctile[c] = t;
    w.cfine[c] = f;
    w.cw[c] = nf;
    if (c == kWideBuckets - 1) {
        w.cbase[c + 1] = b + n;
        w.ctile[c + 1] = t + tiles;
        w.cfine[c + 1] = f + nf;
    }
    for (int i = c; i < 2 * kDirectMaxP * kDirectMaxP; i += kWideBuckets) w.tally[i] = 0;
}

// off[c][t] and loc[c][t] for 64 tiles and 64 buckets: a wave per 16 buckets,
// a lane per tile (prefix over the lanes); also the level 1 tile that holds
// the first record of every level 2 tile
__global__ __launch_bounds__(256) void wide_offsets_kernel(WideWork w) {
    __shared__ uint16_t s_ex[64][66];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int64_t t0 = (int64_t)blockIdx.x * 64;
    const int c0 = blockIdx.y * 64, nc = min(64, w.W - c0);
    for (int i = tid; i < 64 * 65; i += 256) {
        const int t = i / 65, c = i % 65;
        s_ex[t][c] = t0 + t < w.nt && c <= nc ? w.ex1[(t0 + t) * kWideStride + c0 + c] : (uint16_t)0;
    }
    __syncthreads();
    for (int q = 0; q < 16; q++) {
        const int c = wave * 16 + q;
        if (c >= nc) break;
        const uint32_t l = s_ex[lane][c];
        const uint32_t n = s_ex[lane][c + 1] - l;
        const uint32_t o = w.part[(int64_t)blockIdx.x * kWideBuckets + c0 + c] + incl_scan_u32(n) - n;
        const int64_t at = (int64_t)(c0 + c) * w.ntpad + t0 + lane;
        w.off[at] = o;
        w.loc[at] = (uint16_t)l;
        const uint32_t k = (o + kWideTile - 1) / kWideTile;
        if (n > 0 && k * kWideTile < o + n) w.first[w.ctile[c0 + c] + k] = (uint32_t)(t0 + lane);
    }
}

// ---------------------------------------------------------------------------
// Fine boundaries: up to 4096 keys of a coarse bucket, one in each of as many
// equal parts of it (sample_pos), sorted in LDS by a bitonic network.
template <int RW, bool SEG>
__global__ __launch_bounds__(1024) void wide_sample_kernel(const uint32_t* __restrict__ src, LKey lk, WideWork w) {
    constexpr int I = kWideSamples / 1024;
    __shared__ uint64_t s_k[kWideSamples];
    __shared__ uint64_t s_raw[kWideBuckets];
    const int c = blockIdx.x, tid = threadIdx.x;
    const int nw = (int)w.cw[c];
    if (w.lists[5] || nw <= 1) return;
    const uint32_t n = w.tot[c], m = min((uint32_t)kWideSamples, n);
    uint32_t pos[I], at[I];
#pragma unroll
    for (int k = 0; k < I; k++) {
        const uint32_t u = min((uint32_t)(k * 1024 + tid), m - 1);
        pos[k] = (uint32_t)sample_pos(u, m, n);
        at[k] = w.cbase[c] + pos[k];
    }
    if constexpr (!SEG) {
        // the level 1 tile of each position: off[lo] <= pos < off[hi]
        const uint32_t* off = w.off + (int64_t)c * w.ntpad;
        const uint16_t* loc = w.loc + (int64_t)c * w.ntpad;
        const uint32_t t0 = w.ctile[c], t1 = w.ctile[c + 1];
        uint32_t lo[I], hi[I];
#pragma unroll
        for (int k = 0; k < I; k++) {
            const uint32_t t = t0 + pos[k] / kWideTile;
            lo[k] = w.first[t];
            hi[k] = t + 1 < t1 ? w.first[t + 1] + 1 : (uint32_t)w.nt;
        }
        for (;;) {
            bool more = false;
#pragma unroll
            for (int k = 0; k < I; k++) {
                if (hi[k] - lo[k] > 1) {
                    const uint32_t mid = (lo[k] + hi[k]) >> 1;
                    if (off[mid] <= pos[k]) lo[k] = mid; else hi[k] = mid;
                    more = true;
                }
            }
            if (!more) break;
        }
#pragma unroll
        for (int k = 0; k < I; k++) at[k] = w.tile_beg[lo[k]] + loc[lo[k]] + (pos[k] - off[lo[k]]);
    }
#pragma unroll
    for (int k = 0; k < I; k++) {
        uint32_t r[RW];
        RecIO<RW>::load(src, (int64_t)at[k], r);
        s_k[k * 1024 + tid] = (uint32_t)(k * 1024 + tid) < m ? lkey<RW>(r, lk) : ~0ull;
    }
    __syncthreads();
    for (int size = 2; size <= kWideSamples; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
#pragma unroll
            for (int k = 0; k < I / 2; k++) {
                const int p = k * 1024 + tid;
                const int i = 2 * p - (p & (stride - 1)), j = i + stride;
                const uint64_t a = s_k[i], b = s_k[j];
                if ((a > b) == ((i & size) == 0)) {
                    s_k[i] = b;
                    s_k[j] = a;
                }
            }
            __syncthreads();
        }
    }
    if (tid < nw - 1) s_raw[tid] = s_k[(uint32_t)(tid + 1) * m / (uint32_t)nw - 1];
    __syncthreads();
    if (tid < kWideBuckets) w.tables2[(int64_t)c * kWideBuckets + tid] = wide_boundary(s_raw, tid, nw - 1);
}

// The groups of a coarse bucket, a thread per fine bucket: greedy runs of
// neighbouring fine buckets of together at most kWideCap records (their runs
// are adjacent in every tile).  A bucket above that, and one of a single key
// value and more than kWideAlone records (its order is final as it stands),
// is a group by itself.  The greedy run that starts at each bucket comes from
// a search of the prefix; the runs actually taken are marked by pointer
// jumping from bucket 0.  Buckets of 1843 records on average, each sorted by
// itself, left 40% of the sorting workgroups' 3072 slots empty and listed the
// largest; groups of buckets of 1024 fill 83%.  The sorts of 2^28 x 16 B
// clustered keys: 4.1 -> 3.7 ms; of 10,000,019 x 8 B Zipf keys 380 -> 280 us.
// Buckets of 512 fill 92%, but the level's search and ballots then cost what
// the sort gains (2^26 records in 2000 segments: 449 + 672 us instead of
// 407 + 692).
// Also the copy tasks of the one-value buckets above the in-LDS capacity and
// of the oversized ones, which are listed.
constexpr uint32_t kWideAlone = 64;
__global__ __launch_bounds__(kWideBuckets) void wide_fine_kernel(WideWork w) {
    __shared__ uint32_t s_tmp[kWWaves];
    __shared__ uint32_t s_pref[kWideBuckets + 1];
    __shared__ uint16_t s_jump[2][kWideBuckets + 1];
    __shared__ uint8_t s_mark[kWideBuckets + 1];
    __shared__ uint64_t s_alone[kWWaves];
    __shared__ uint32_t s_id;
    const int c = blockIdx.x, f = threadIdx.x, wave = f >> 6, lane = f & 63;
    const int nw = (int)w.cw[c];
    if (w.lists[5] || nw == 0) return;
    const uint32_t t0 = w.ctile[c];
    const int nt = (int)(w.ctile[c + 1] - t0);
    uint32_t sum = 0;
    if (f < nw) {
        constexpr int U = 8;
        for (int q0 = 0; q0 < nt; q0 += U) {
            uint32_t a[U], b[U];
#pragma unroll
            for (int q = 0; q < U; q++) {
                const uint16_t* ex = w.ex2 + (int64_t)(t0 + min(q0 + q, nt - 1)) * kWideStride;
                a[q] = ex[f];
                b[q] = ex[f + 1];
            }
#pragma unroll
            for (int q = 0; q < U; q++) sum += q0 + q < nt ? b[q] - a[q] : 0u;
        }
    }
    const uint32_t pre = scan_block<kWideBuckets>(sum, s_tmp);
    const bool single = f < nw && wide_single(w.tables2 + (int64_t)c * kWideBuckets, f, nw - 1);
    const uint32_t most = min((uint32_t)kWideCap, w.cap);  // records of a group of several
    const bool alone = sum > most || (single && sum > kWideAlone);
    const uint64_t am = __ballot(alone);
    if (lane == 0) s_alone[wave] = am;
    s_pref[f] = pre;
    s_mark[f] = f == 0 ? 1 : 0;
    if (f == kWideBuckets - 1) {
        s_pref[kWideBuckets] = pre + sum;
        s_mark[kWideBuckets] = 0;
        s_jump[0][kWideBuckets] = s_jump[1][kWideBuckets] = (uint16_t)kWideBuckets;
    }
    __syncthreads();
    int fe = f + 1;
    if (!alone && f < nw) {
        // up to the next bucket that stands alone
        int stop = nw;
        for (int q = wave; q < kWWaves; q++) {
            const uint64_t m = q == wave ? (lane == 63 ? 0 : s_alone[q] >> (lane + 1) << (lane + 1)) : s_alone[q];
            if (m) {
                stop = q * 64 + __builtin_ctzll(m);
                break;
            }
        }
        // the largest fe <= stop with pref[fe] - pref[f] <= most
        int lo = f + 1, hi = stop;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (s_pref[mid] - pre <= most) lo = mid; else hi = mid - 1;
        }
        fe = lo;
    }
    s_jump[0][f] = (uint16_t)(f < nw ? (fe < nw ? fe : kWideBuckets) : kWideBuckets);
    __syncthreads();
    int cur = 0;
    for (int k = 1; k < nw; k <<= 1, cur ^= 1) {
        const int j = s_jump[cur][f];
        const bool m = s_mark[f];
        s_jump[cur ^ 1][f] = s_jump[cur][j];
        __syncthreads();
        if (m) s_mark[j] = 1;
        __syncthreads();
    }
    const uint32_t cnt = f < nw && s_mark[f] ? s_pref[fe] - pre : 0u;
    const uint32_t idx = scan_block<kWideBuckets>(cnt ? 1u : 0u, s_tmp);
    if (f == kWideBuckets - 1) s_id = atomicAdd(&w.lists[6], idx + (cnt ? 1u : 0u));
    __syncthreads();
    if (cnt == 0) return;
    const uint32_t id = s_id + idx;
    const uint32_t base = w.cbase[c] + pre;
    w.fcnt[id] = cnt;
    w.fbase[id] = base;
    w.desc[id] = WideBucket{t0, w.cbase[c], (uint16_t)nt, (uint16_t)f, (uint16_t)fe, 0};
    // (many one-value groups) sorted with the listed ones
    if (id >= (uint32_t)w.ngrid && cnt <= w.cap) w.medium[atomicAdd(&w.lists[2], 1u)] = id;
    if (cnt > w.cap) {
        if (!single) {
            const uint32_t slot = atomicAdd(&w.lists[0], 1u);
            if ((int)slot < w.max_overflow) {
                w.overflow[2 * slot] = base;
                w.overflow[2 * slot + 1] = cnt;
            }
        }
        const uint32_t k = (cnt + kWideCopy - 1) / kWideCopy;
        const uint32_t at = atomicAdd(&w.lists[4], k);
        for (uint32_t q = 0; q < k; q++)
            if (at + q < (uint32_t)w.ncopy) w.copy[at + q] = make_uint2(id, q * kWideCopy);
    }
}

// ---------------------------------------------------------------------------
// Splitters and counts.  A level 2 tile of the coarse bucket that holds a
// splitter: its records below the splitter and at most equal to it, by rank
// (a tile's records come rank by rank, so a wave's lanes mostly share one).
template <int RW>
__global__ __launch_bounds__(kWBlock) void wide_tally_kernel(const uint32_t* __restrict__ out,
                                                             const uint32_t* __restrict__ part, LKey lk, int P,
                                                             const int64_t* __restrict__ C,
                                                             const int64_t* __restrict__ begin, WideWork w) {
    __shared__ WideRunTab s_rt;
    __shared__ uint32_t s_tmp[2 * (kWWaves + 1)];
    __shared__ uint32_t s_lt[kDirectMaxP], s_le[kDirectMaxP];
    __shared__ uint32_t s_begin[kDirectMaxP];
    const int i = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if (w.lists[5]) return;
    const int64_t Ci = C[i + 1];
    uint32_t r[RW];
    RecIO<RW>::load(out, Ci > 0 ? Ci - 1 : 0, r);
    const uint64_t v = lkey<RW>(r, lk);
    const uint64_t m = __ballot(tid < w.W - 1 && w.tables[tid] < v);
    if (lane == 0) s_tmp[wave] = (uint32_t)__popcll(m);
    if (tid < kDirectMaxP) {
        s_lt[tid] = s_le[tid] = 0;
        s_begin[tid] = tid < P ? (uint32_t)begin[tid] : 0xffffffffu;
    }
    __syncthreads();
    int c = 0;
#pragma unroll
    for (int q = 0; q < kWWaves; q++) c += (int)s_tmp[q];
    const uint32_t t0 = w.ctile[c], tile = t0 + blockIdx.x;
    if (w.cw[c] == 0 || tile >= w.ctile[c + 1]) return;
    __syncthreads();
    const uint32_t p0 = blockIdx.x * (uint32_t)kWideTile;
    const uint32_t cnt = min((uint32_t)kWideTile, w.tot[c] - p0);
    wide_locate(w, c, tile, p0, p0 + cnt, s_rt, s_tmp);
    constexpr int U = 4;
    for (int k0 = 0; k0 < kWItems; k0 += U) {
        uint32_t rr[U][RW], at[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            at[u] = s_rt.at(min((uint32_t)(wave * kWSpan + (k0 + u) * 64 + lane), cnt - 1));
            RecIO<RW>::load(part, (int64_t)at[u], rr[u]);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const bool in = (uint32_t)(wave * kWSpan + (k0 + u) * 64 + lane) < cnt;
            const uint64_t key = lkey<RW>(rr[u], lk);
            // the last rank that begins at or before the record (empty ranks
            // before it begin there too)
            int j = 0;
#pragma unroll
            for (int step = kDirectMaxP / 2; step > 0; step >>= 1) j += s_begin[j + step] <= at[u] ? step : 0;
            const bool lt = in && key < v, le = in && key <= v;
            const int j0 = __builtin_amdgcn_readfirstlane(j);
            if (__ballot(j != j0) == 0) {
                const uint64_t ml = __ballot(lt), me = __ballot(le);
                if (lane == 0 && me) {
                    atomicAdd(&s_lt[j0], (uint32_t)__popcll(ml));
                    atomicAdd(&s_le[j0], (uint32_t)__popcll(me));
                }
            } else {
                if (lt) atomicAdd(&s_lt[j], 1u);
                if (le) atomicAdd(&s_le[j], 1u);
            }
        }
    }
    __syncthreads();
    if (tid < P && s_le[tid]) {
        uint32_t* t = w.tally + 2 * (i * kDirectMaxP + tid);
        if (s_lt[tid]) atomicAdd(t, s_lt[tid]);
        atomicAdd(t + 1, s_le[tid]);
    }
}

// Block j: rank j's records below every splitter, from its records in the
// coarse buckets before the splitter's and the tally of that bucket.  The
// block that finishes last solves the layout.
template <int RW>
__global__ __launch_bounds__(1024) void wide_counts_kernel(const uint32_t* __restrict__ out, LKey lk, int P, int64_t n,
                                                           DirectWork d, WideWork w, DirectResult* __restrict__ res) {
    constexpr int BLOCK = 1024, NW = BLOCK / 64;
    __shared__ uint64_t s_tab[kWideBuckets];
    __shared__ uint32_t s_pref[BLOCK], s_mine[BLOCK];
    __shared__ uint32_t s_tmp[NW];
    __shared__ uint32_t s_c[kDirectMaxP + 1][kDirectMaxP];
    __shared__ uint32_t s_err;
    __shared__ int s_last;
    const int j = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int P1 = P + 1;
    if (tid == 0) s_err = 0;
    bool hit = false;
    if (P > 1 && !w.lists[5]) {
        if (tid < kWideBuckets) s_tab[tid] = w.tables[tid];
        uint32_t mine = 0;
        if (tid < w.W) {
            const uint32_t* off = w.off + (int64_t)tid * w.ntpad;
            mine = off[d.tile_start[j + 1]] - off[d.tile_start[j]];
        }
        s_mine[tid] = mine;
        s_pref[tid] = scan_block<BLOCK>(mine, s_tmp);
        __syncthreads();
        if (tid < P - 1) {
            const int64_t Ci = d.C[tid + 1];
            uint32_t r[RW];
            RecIO<RW>::load(out, Ci > 0 ? Ci - 1 : 0, r);
            const uint64_t v = lkey<RW>(r, lk);
            hit = d.prop && Ci > 0 && d.prop[tid] == v;
            int b = 0;
            for (int step = kWideBuckets / 2; step > 0; step >>= 1) b += s_tab[b + step - 1] < v ? step : 0;
            b = min(b, w.W - 1);
            const uint32_t* t = w.tally + 2 * (tid * kDirectMaxP + j);
            const bool one = w.cw[b] == 0;
            const uint32_t lt = s_pref[b] + (one ? 0u : t[0]);
            const uint32_t le = s_pref[b] + (one ? s_mine[b] : t[1]);
            d.myclt[(int64_t)j * P1 + tid + 1] = lt;
            d.mycle[(int64_t)j * P1 + tid + 1] = le;
            store_agent(d.cross + tid * kDirectMaxP + j, ((uint64_t)le << 32) | lt);
            if (j == 0) {
                d.split[4 * tid] = v;
                d.split[4 * tid + 1] = d.split[4 * tid + 2] = d.split[4 * tid + 3] = 0;
            }
        } else if (j == 0 && tid >= BLOCK - 2) {
            uint32_t r[RW];
            const int q = tid - (BLOCK - 2);
            RecIO<RW>::load(out, q ? n - 1 : 0, r);
            d.pminmax[4 * q] = lkey<RW>(r, lk);
            for (int k = 1; k < 4; k++) d.pminmax[4 * q + k] = 0;
        }
        // the block's agent-scope stores to cross are complete before it is
        // counted
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0)
            s_last = __hip_atomic_fetch_add(&w.lists[7], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) ==
                     (uint32_t)(P - 1);
        __syncthreads();
        if (!s_last) return;
        if (tid == 0) w.lists[7] = 0;  // the counts may run again in this call
        if (tid < kDirectMaxP) s_c[0][tid] = 0;
        const uint32_t cnt = lane < P ? (uint32_t)d.count[lane] : 0u;
        if (tid < P) {
            d.myC[(int64_t)tid * P1] = 0;
            d.myclt[(int64_t)tid * P1] = d.mycle[(int64_t)tid * P1] = 0;
            d.myclt[(int64_t)tid * P1 + P] = d.mycle[(int64_t)tid * P1 + P] = d.count[tid];
        }
        solve_layout<NW>(P, d, d.C, &s_err, s_c, [&](int r, uint32_t& a, uint32_t& e) {
            const uint64_t x = r < P - 1 ? load_agent(d.cross + r * kDirectMaxP + lane) : ((uint64_t)cnt << 32) | cnt;
            a = (uint32_t)x;
            e = (uint32_t)(x >> 32);
        });
    } else if (j > 0) {
        return;
    }
    __syncthreads();
    const uint64_t hits = __ballot(hit);  // splitters belong to the first wave
    if (tid == 0) res->exact = (uint32_t)__popcll(hits);
    if (tid < 3) res->lists[tid] = w.lists[tid];
    if (tid == 3) res->lists[3] = w.lists[5];
    if (tid < 2) res->sums[tid] = d.checksum[tid];
    if (tid == 2) res->err = d.err[0] | s_err;
    if (tid == 3) res->buckets = w.cfine[w.W];
}

// ---------------------------------------------------------------------------
int launch_wide_level1(int rw, const void* src, void* dst, const LKey& lk, const SegDev& sd, const WideWork& w,
                       long long* checksum, hipStream_t st) {
    const uint32_t* s = (const uint32_t*)src;
    uint32_t* o = (uint32_t*)dst;
    const dim3 g((unsigned)w.nt), b(kWBlock);
    if (rw == 2) hipLaunchKernelGGL((wide_part_kernel<2, kLevel1>), g, b, 0, st, s, o, nullptr, lk, sd, w, checksum);
    else if (rw == 4) hipLaunchKernelGGL((wide_part_kernel<4, kLevel1>), g, b, 0, st, s, o, nullptr, lk, sd, w, checksum);
    else return -1;
    MPSG_CHECK(hipGetLastError());
    // off and loc have an entry past the last tile (the bucket's total)
    const int64_t rows = (w.nt + 64) / 64;
    const unsigned cb = (unsigned)((w.W + 63) / 64);
    hipLaunchKernelGGL(wide_sums_kernel, dim3((unsigned)rows), dim3(kWideBuckets), 0, st, w);
    MPSG_CHECK(hipGetLastError());
    hipLaunchKernelGGL(wide_scan_kernel, dim3(cb), dim3(1024), 0, st, w, rows);
    MPSG_CHECK(hipGetLastError());
    hipLaunchKernelGGL(wide_plan_kernel, dim3(1), dim3(kWideBuckets), 0, st, w);
    MPSG_CHECK(hipGetLastError());
    hipLaunchKernelGGL(wide_offsets_kernel, dim3((unsigned)rows, cb), dim3(256), 0, st, w);
    MPSG_CHECK(hipGetLastError());
    if (rw == 2) hipLaunchKernelGGL((wide_sample_kernel<2, false>), dim3((unsigned)w.W), dim3(1024), 0, st, o, lk, w);
    else hipLaunchKernelGGL((wide_sample_kernel<4, false>), dim3((unsigned)w.W), dim3(1024), 0, st, o, lk, w);
    MPSG_CHECK(hipGetLastError());
    return 0;
}

int launch_wide_level2(int rw, const void* src, void* dst, void* out, const LKey& lk, const WideWork& w,
                       long long* checksum_out, hipStream_t st) {
    const uint32_t* s = (const uint32_t*)src;
    uint32_t *d = (uint32_t*)dst, *o = (uint32_t*)out;
    const dim3 g((unsigned)w.nt2), b(kWBlock);
    const SegDev none{nullptr, nullptr, nullptr, 0, 0};
    if (rw == 2) hipLaunchKernelGGL((wide_part_kernel<2, kLevel2>), g, b, 0, st, s, d, o, lk, none, w, checksum_out);
    else if (rw == 4) hipLaunchKernelGGL((wide_part_kernel<4, kLevel2>), g, b, 0, st, s, d, o, lk, none, w, checksum_out);
    else return -1;
    MPSG_CHECK(hipGetLastError());
    hipLaunchKernelGGL(wide_fine_kernel, dim3((unsigned)w.W), dim3(kWideBuckets), 0, st, w);
    MPSG_CHECK(hipGetLastError());
    return 0;
}

int launch_wide_segments(int rw, const void* src, void* tmp, void* out, const LKey& lk, const WideWork& w,
                         hipStream_t st) {
    const uint32_t* s = (const uint32_t*)src;
    uint32_t* t = (uint32_t*)tmp;
    const dim3 g((unsigned)w.nt2), b(kWBlock), gw((unsigned)w.W);
    const SegDev none{nullptr, nullptr, nullptr, 0, 0};
    int rc = 0;
    if (rw != 2 && rw != 4) return -1;
    if ((rc = launch_fill_u32(w.lists, 0u, 8, st))) return rc;
    if (rw == 2) hipLaunchKernelGGL((wide_sample_kernel<2, true>), gw, dim3(1024), 0, st, s, lk, w);
    else hipLaunchKernelGGL((wide_sample_kernel<4, true>), gw, dim3(1024), 0, st, s, lk, w);
    MPSG_CHECK(hipGetLastError());
    if (rw == 2) hipLaunchKernelGGL((wide_part_kernel<2, kSegment>), g, b, 0, st, s, t, nullptr, lk, none, w, nullptr);
    else hipLaunchKernelGGL((wide_part_kernel<4, kSegment>), g, b, 0, st, s, t, nullptr, lk, none, w, nullptr);
    MPSG_CHECK(hipGetLastError());
    hipLaunchKernelGGL(wide_fine_kernel, gw, dim3(kWideBuckets), 0, st, w);
    MPSG_CHECK(hipGetLastError());
    if ((rc = launch_wide_sort(rw, tmp, out, lk, w, nullptr, st))) return rc;
    return launch_wide_big(rw, out, tmp, lk, w, st);
}

int launch_wide_counts(int rw, const void* out, const void* part, const LKey& lk, const DirectShape& sh,
                       const DirectWork& d, const WideWork& w, DirectResult* res, hipEvent_t stop, hipStream_t st) {
    const uint32_t *o = (const uint32_t*)out, *p = (const uint32_t*)part;
    if (rw != 2 && rw != 4) return -1;
    if (sh.P > 1) {
        const dim3 g(kWideRuns, (unsigned)(sh.P - 1)), b(kWBlock);
        if (rw == 2) hipLaunchKernelGGL(wide_tally_kernel<2>, g, b, 0, st, o, p, lk, sh.P, d.C, d.begin, w);
        else hipLaunchKernelGGL(wide_tally_kernel<4>, g, b, 0, st, o, p, lk, sh.P, d.C, d.begin, w);
        MPSG_CHECK(hipGetLastError());
    }
    const dim3 g((unsigned)sh.P), b(1024);
    if (rw == 2) hipExtLaunchKernelGGL(wide_counts_kernel<2>, g, b, 0, st, nullptr, stop, 0, o, lk, sh.P, sh.n, d, w, res);
    else hipExtLaunchKernelGGL(wide_counts_kernel<4>, g, b, 0, st, nullptr, stop, 0, o, lk, sh.P, sh.n, d, w, res);
    MPSG_CHECK(hipGetLastError());
    return 0;
}

}  // namespace mpsg
