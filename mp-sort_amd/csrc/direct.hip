// direct.hip -- the sort of up to 64 ranks without per-rank local sorts: the
// records of all ranks are partitioned into key buckets (boundaries from a
// sorted sample), every bucket is sorted in LDS into the output, and the
// splitters and counts of the histogram sort (mpsort-mpi.c:375-510) are read
// off the result.  The reference's FirstSort, exchange and SecondSort
// (mpsort-mpi.c:369,571-597) produce that same stable order.
#include <hip/hip_ext.h>

#include <algorithm>

#include "direct.h"
#include "layout_dev.h"
#include "lsort_dev.h"

namespace mpsg {

// ---------------------------------------------------------------------------
// Sample.  Block c takes the keys at positions sample_pos(u), u = 1024 c ..
// 1024 c + 1023, and sorts them: one key per thread, a bitonic network whose
// strides below 64 are lane exchanges and whose ten larger ones go through
// LDS.  Block 0 also writes the call's tables and clears its counters (every
// later kernel of the call reads them).
__device__ __forceinline__ uint64_t bitonic1024(uint64_t v, uint64_t* s_k) {
    const int tid = threadIdx.x;
    for (int size = 2; size <= kDirectChunk; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            uint64_t o;
            if (stride >= 64) {
                s_k[tid] = v;
                __syncthreads();
                o = s_k[tid ^ stride];
                __syncthreads();
            } else {
                o = __shfl_xor(v, stride, 64);
            }
            const bool lower = (tid & stride) == 0, up = (tid & size) == 0;
            v = (lower == up) ? (o < v ? o : v) : (o > v ? o : v);
        }
    }
    return v;
}

// boundary q (1 .. W - 1) is the smallest sample rank r with (r + 1) W >= q S
__device__ __forceinline__ void put_boundary(uint64_t key, int rank, int S, int W, uint64_t* raw) {
    const int64_t x = (int64_t)(rank + 1) * W;
    const int q = (int)(x / S);
    if (q >= 1 && q < W && x - (int64_t)q * S < W) raw[q - 1] = key;
}

template <int RW>
__global__ __launch_bounds__(kDirectChunk) void direct_sample_kernel(const uint32_t* __restrict__ src, LKey lk,
                                                                     DirectShape sh, DirectWork w,
                                                                     int clear_sums) {
    __shared__ uint64_t s_k[kDirectChunk];
    const int tid = threadIdx.x;
    if (blockIdx.x == 0) {
        if (tid <= sh.P) {
            w.C[tid] = sh.C[tid];
            w.tile_start[tid] = sh.tile_start[tid];
            if (tid < sh.P) {
                w.begin[tid] = sh.begin[tid];
                w.count[tid] = sh.begin[tid + 1] - sh.begin[tid];
            }
        }
        if (tid < 8) w.lists[tid] = 0;
        if (tid < 4) w.err[tid] = 0;
        if (tid < 2 && clear_sums) w.checksum[tid] = 0;
    }
    if (sh.S == 0) return;  // the boundaries come from elsewhere
    const int64_t u = (int64_t)blockIdx.x * kDirectChunk + tid;
    const int64_t pos = (int64_t)sample_pos((uint32_t)u, (uint32_t)sh.S, (uint64_t)sh.n);
    uint32_t r[RW];
    RecIO<RW>::load(src, pos, r);
    const uint64_t v = bitonic1024(lkey<RW>(r, lk), s_k);
    if (sh.S == kDirectChunk) put_boundary(v, tid, sh.S, sh.W, w.raw);
    else w.chunks[u] = v;
}

// The rank of every sample key among all chunks (equal keys in chunk order):
// its index in its own chunk plus a binary search in each other chunk, 16
// chunks staged in LDS at a time so that 16 searches advance together
// (8 loads of a thread in flight while a stage is copied in).
constexpr int kRankBlock = 256, kRankStage = 16;
__global__ __launch_bounds__(kRankBlock) void direct_rank_kernel(int S, int W, const uint64_t* __restrict__ chunks,
                                                                 uint64_t* __restrict__ raw) {
    __shared__ __attribute__((aligned(16))) uint64_t s_k[kRankStage * kDirectChunk];
    const int nch = S / kDirectChunk, tid = threadIdx.x;
    const int g = blockIdx.x * kRankBlock + tid;
    const int mine = g / kDirectChunk;
    const uint64_t key = chunks[g];
    int rank = g % kDirectChunk;
    for (int c0 = 0; c0 < nch; c0 += kRankStage) {
        const int m = min(kRankStage, nch - c0);
        __syncthreads();
        const uint4* from = reinterpret_cast<const uint4*>(chunks + (int64_t)c0 * kDirectChunk);
        uint4* to = reinterpret_cast<uint4*>(s_k);
        constexpr int U = 8;
        const int words = m * kDirectChunk / 2;  // a multiple of kRankBlock
        for (int i = tid; i < words; i += U * kRankBlock) {
            uint4 x[U];
#pragma unroll
            for (int u = 0; u < U; u++) x[u] = from[min(i + u * kRankBlock, words - 1)];
#pragma unroll
            for (int u = 0; u < U; u++)
                if (i + u * kRankBlock < words) to[i + u * kRankBlock] = x[u];
        }
        __syncthreads();
        int lo[kRankStage];
#pragma unroll
        for (int c = 0; c < kRankStage; c++) lo[c] = 0;
#pragma unroll
        for (int step = kDirectChunk / 2; step > 0; step >>= 1) {
#pragma unroll
            for (int c = 0; c < kRankStage; c++) {
                if (c < m) {
                    const uint64_t x = s_k[c * kDirectChunk + lo[c] + step - 1];
                    // chunks before this one: #{<= key}; after it: #{< key}
                    if (c0 + c < mine ? x <= key : x < key) lo[c] += step;
                }
            }
        }
#pragma unroll
        for (int c = 0; c < kRankStage; c++) {
            if (c < m && c0 + c != mine) {
                const uint64_t x = s_k[c * kDirectChunk + lo[c]];
                rank += lo[c] + ((c0 + c < mine ? x <= key : x < key) ? 1 : 0);
            }
        }
    }
    put_boundary(key, rank, S, W, raw);
}

// ---------------------------------------------------------------------------
// Bucket of every record and the tiles' bucket counts.  The boundary table is
// made from the raw sample keys by every block (block 0 keeps it): where
// boundaries repeat a key v, the first of them becomes v - 1, so that
// (v - 1, v] holds that key alone; entries past W - 2 are the largest key.
// The searches of a thread's U records advance together.
template <int RW>
__global__ __launch_bounds__(512) void direct_hist_kernel(const uint32_t* __restrict__ src, SegDev seg, int64_t ntiles,
                                                          int64_t tpb, int tile_recs, LKey lk, int W, int step0,
                                                          const uint64_t* __restrict__ raw,
                                                          uint64_t* __restrict__ tables,
                                                          uint16_t* __restrict__ tile_cnt, uint16_t* __restrict__ bkt,
                                                          long long* __restrict__ checksum) {
    constexpr int BLOCK = 512, U = RW == 2 ? 4 : 3;
    __shared__ uint64_t s_tab[kLBins];
    __shared__ uint32_t s_th[kLBins];
    __shared__ long long s_sum[BLOCK / 64];
    const int tid = threadIdx.x;
    for (int e = tid; e < kLBins; e += BLOCK) {
        uint64_t t = ~0ull;
        if (e < W - 1) {
            const uint64_t v = raw[e];
            const bool first = e == 0 || raw[e - 1] < v;
            const bool repeated = e + 1 < W - 1 && raw[e + 1] == v;
            t = first && repeated && v > 0 ? v - 1 : v;
        }
        s_tab[e] = t;
        s_th[e] = 0;
        if (blockIdx.x == 0 && e < kLBounds) tables[e] = t;
    }
    __syncthreads();
    const int64_t t0 = (int64_t)blockIdx.x * tpb, t1 = min(ntiles, t0 + tpb);
    long long csum = 0;
    for (int64_t tile = t0; tile < t1; tile++) {
        const int s = seg_of_tile(seg, tile);
        const int64_t sbeg = seg.begin[s];
        const int64_t begin = sbeg + (tile - seg.tile_start[s]) * tile_recs;
        const int64_t end = min(sbeg + seg.count[s], begin + (int64_t)tile_recs);
        for (int64_t i0 = begin + tid; i0 < end; i0 += U * BLOCK) {
            uint32_t r[U][RW];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int64_t i = i0 + (int64_t)u * BLOCK;
                RecIO<RW>::load(src, i < end ? i : end - 1, r[u]);
            }
            uint64_t k[U];
            int lo[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                k[u] = lkey<RW, true>(r[u], lk);
                lo[u] = 0;
            }
            for (int step = step0; step > 0; step >>= 1) {
                uint64_t v[U];
#pragma unroll
                for (int u = 0; u < U; u++) v[u] = s_tab[min(lo[u] + step - 1, kLBounds)];
#pragma unroll
                for (int u = 0; u < U; u++) lo[u] += (v[u] < k[u] && lo[u] + step <= kLBounds) ? step : 0;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int64_t i = i0 + (int64_t)u * BLOCK;
                if (i < end) {
                    if (checksum) {
#pragma unroll
                        for (int q = 0; q < RW; q++) csum += sbyte_sum(r[u][q]);
                    }
                    bkt[i] = (uint16_t)lo[u];
                    atomicAdd(&s_th[lo[u]], 1u);
                }
            }
        }
        __syncthreads();
        for (int b = tid; b < kLBins; b += BLOCK) {
            tile_cnt[tile * kLBins + b] = (uint16_t)s_th[b];
            s_th[b] = 0;
        }
        __syncthreads();
    }
    if (checksum) {
        csum = wave_sum_ll(csum);
        if ((tid & 63) == 0) s_sum[tid >> 6] = csum;
        __syncthreads();
        if (tid == 0) {
            long long a = 0;
            for (int q = 0; q < BLOCK / 64; q++) a += s_sum[q];
            atomicAdd((unsigned long long*)checksum, (unsigned long long)a);
        }
    }
}

// tile_off[t][b] = bucket b's records in the tiles before t, and the totals:
// a block per 64 buckets, its 16 waves over equal runs of tiles (counts
// summed, prefixed over the waves, then walked again)
__global__ __launch_bounds__(1024) void direct_scan_kernel(const uint16_t* __restrict__ tile_cnt, int64_t ntiles,
                                                           uint32_t* __restrict__ tile_off, uint32_t* __restrict__ tot) {
    __shared__ uint32_t s_part[16][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int b = blockIdx.x * 64 + lane;
    const int64_t per = (ntiles + 15) / 16;
    const int64_t t0 = min(ntiles, wave * per), t1 = min(ntiles, t0 + per);
    constexpr int U = 16;
    uint32_t sum = 0;
    for (int64_t t = t0; t < t1; t += U) {
        uint32_t c[U];
#pragma unroll
        for (int q = 0; q < U; q++) c[q] = t + q < t1 ? tile_cnt[(t + q) * kLBins + b] : 0u;
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
    if (wave == 0) tot[b] = all;
    for (int64_t t = t0; t < t1; t += U) {
        uint32_t c[U];
#pragma unroll
        for (int q = 0; q < U; q++) c[q] = t + q < t1 ? tile_cnt[(t + q) * kLBins + b] : 0u;
#pragma unroll
        for (int q = 0; q < U; q++) {
            if (t + q < t1) tile_off[(t + q) * kLBins + b] = run;
            run += c[q];
        }
    }
}

// ---------------------------------------------------------------------------
// Splitters, counts and layout.  Splitter i = key of output record C[i+1] - 1
// (the smallest key when C[i+1] is 0, where the reference's bisection ends).
// Block j counts rank j's records below every splitter: its records in the
// buckets before the splitter's (a prefix over the buckets of its tiles'
// offsets: a rank's run in a bucket starts where its first tile's does), plus
// those of its run in that bucket that are smaller (or equal), a wave per
// splitter.  The block that finishes last solves the layout
// (_solve_for_layout_mpi mpsort-mpi.c:663-727): a wave per receiver, a lane
// per sender (the greedy fill from sender 0 as a prefix over the senders'
// supplies), then the send counts and the call's results.  Block j reads two
// rows of offsets; a block per splitter, which read 2 P rows each, took 43
// instead of 12 us at 64 ranks, and the layout in a launch of its own 13 more.
template <int RW>
__global__ __launch_bounds__(1024) void direct_counts_kernel(const uint32_t* __restrict__ out,
                                                             const uint32_t* __restrict__ part, LKey lk, int P,
                                                             int64_t n, int64_t ntiles, DirectWork w,
                                                             DirectResult* __restrict__ res) {
    constexpr int BLOCK = 1024, NW = BLOCK / 64, Q = kDirectMaxP / NW;  // splitters (receivers) per wave
    __shared__ uint64_t s_tab[kLBins];
    __shared__ uint32_t s_pref[kLBins];
    __shared__ uint32_t s_tmp[NW];
    __shared__ uint64_t s_v[kDirectMaxP];
    __shared__ int s_b[kDirectMaxP];
    __shared__ uint32_t s_c[kDirectMaxP + 1][kDirectMaxP];  // [receiver edge][sender]
    __shared__ uint32_t s_err;
    __shared__ int s_last;
    const int j = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int P1 = P + 1;
    if (tid == 0) s_err = 0;
    if (P > 1) {
        s_tab[tid] = tid < kLBounds ? w.tables[tid] : ~0ull;
        const int64_t ta = w.tile_start[j], tb = w.tile_start[j + 1];
        const uint32_t* oa = w.tile_off + ta * kLBins;
        const uint32_t* ob = tb >= ntiles ? w.tot : w.tile_off + tb * kLBins;
        const uint32_t mine = ta < tb ? ob[tid] - oa[tid] : 0u;
        s_pref[tid] = scan_block<BLOCK>(mine, s_tmp);
        if (tid < P - 1) {
            const int64_t Ci = w.C[tid + 1];
            uint32_t r[RW];
            RecIO<RW>::load(out, Ci > 0 ? Ci - 1 : 0, r);
            const uint64_t v = lkey<RW>(r, lk);
            s_v[tid] = v;
            s_b[tid] = (int)bucket_of(v, s_tab);  // s_tab is complete: scan_block has barriers
            if (j == 0) {
                w.split[4 * tid] = v;
                w.split[4 * tid + 1] = w.split[4 * tid + 2] = w.split[4 * tid + 3] = 0;
            }
        } else if (j == 0 && tid >= BLOCK - 2) {
            uint32_t r[RW];
            const int q = tid - (BLOCK - 2);
            RecIO<RW>::load(out, q ? n - 1 : 0, r);
            w.pminmax[4 * q] = lkey<RW>(r, lk);
            for (int k = 1; k < 4; k++) w.pminmax[4 * q + k] = 0;
        }
        __syncthreads();
        // this wave's splitters: bounds of the runs first, then the records
        uint32_t r0[Q], r1[Q], lt[Q], le[Q];
        int64_t base[Q];
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int i = q * NW + wave;
            r0[q] = r1[q] = lt[q] = le[q] = 0;
            base[q] = 0;
            if (i < P - 1 && ta < tb) {
                const int b = s_b[i];
                r0[q] = oa[b];
                r1[q] = ob[b];
                base[q] = w.base[b];
                lt[q] = le[q] = s_pref[b];
                if (single_bucket(s_tab, b)) {  // the splitter's own key alone: not read
                    le[q] += r1[q] - r0[q];
                    r1[q] = r0[q];
                }
            }
        }
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int i = q * NW + wave;
            const uint64_t v = s_v[min(i, kDirectMaxP - 1)];
            for (uint32_t x = r0[q]; x < r1[q]; x += 64) {
                uint32_t r[RW];
                const bool in = x + lane < r1[q];
                RecIO<RW>::load(part, base[q] + (in ? x + lane : r0[q]), r);
                const uint64_t k = lkey<RW>(r, lk);
                lt[q] += (uint32_t)__popcll(__ballot(in && k < v));
                le[q] += (uint32_t)__popcll(__ballot(in && k <= v));
            }
        }
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int i = q * NW + wave;
            if (i < P - 1 && lane == 0) {
                w.myclt[(int64_t)j * P1 + i + 1] = lt[q];
                w.mycle[(int64_t)j * P1 + i + 1] = le[q];
                store_agent(w.cross + i * kDirectMaxP + j, ((uint64_t)le[q] << 32) | lt[q]);
            }
        }
        // the block's agent-scope stores to cross are complete before it is
        // counted (a fence by every wave would write back its L2 each time)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0)
            s_last = __hip_atomic_fetch_add(&w.lists[7], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) ==
                     (uint32_t)(P - 1);
        __syncthreads();
        if (!s_last) return;
        if (tid == 0) w.lists[7] = 0;  // the counts may run again in this call
        if (tid < kDirectMaxP) s_c[0][tid] = 0;
        const uint32_t cnt = lane < P ? (uint32_t)w.count[lane] : 0u;
        if (tid < P) {
            w.myC[(int64_t)tid * P1] = 0;
            w.myclt[(int64_t)tid * P1] = w.mycle[(int64_t)tid * P1] = 0;
            w.myclt[(int64_t)tid * P1 + P] = w.mycle[(int64_t)tid * P1 + P] = w.count[tid];
        }
        solve_layout<NW>(P, w, w.C, &s_err, s_c, [&](int r, uint32_t& a, uint32_t& e) {
            const uint64_t x = r < P - 1 ? load_agent(w.cross + r * kDirectMaxP + lane) : ((uint64_t)cnt << 32) | cnt;
            a = (uint32_t)x;
            e = (uint32_t)(x >> 32);
        });
    }
    __syncthreads();
    if (tid < 4) res->lists[tid] = w.lists[tid];
    if (tid < 2) res->sums[tid] = w.checksum[tid];
    if (tid == 2) res->err = w.err[0] | s_err;
    if (tid == 3) res->scatter_err = w.err[1];
}

// ---------------------------------------------------------------------------
// The counts of a small sort whose n keys (in input order) and splitter
// values lie in LDS: record e of rank j is below splitter i when i >= #{values
// <= its key}, and at most equal to it when i >= #{values < its key}; one LDS
// count each, prefixed over the splitters (a wave per rank, a lane per
// splitter), then the layout.  The searches of a thread's four records
// advance together.
struct SmallCounts {
    uint32_t lt[kDirectMaxP][kDirectMaxP], le[kDirectMaxP][kDirectMaxP];  // [rank][splitter]
    uint32_t c[kDirectMaxP + 1][kDirectMaxP];
    uint64_t v[kDirectMaxP];
    int begin[kDirectMaxP];
    uint32_t err;
};
template <int BLOCK>
__device__ __forceinline__ void small_counts(const DirectShape& sh, const DirectWork& w, const uint64_t* s_key,
                                             SmallCounts& s) {
    constexpr int NW = BLOCK / 64, Q = kDirectMaxP / NW, U = 4;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int P = sh.P, P1 = P + 1, n = (int)sh.n;
    for (int i = tid; i < kDirectMaxP * kDirectMaxP; i += BLOCK) (&s.lt[0][0])[i] = (&s.le[0][0])[i] = 0;
    if (tid < kDirectMaxP) s.c[0][tid] = 0;
    if (tid < P) s.begin[tid] = (int)sh.begin[tid];
    __syncthreads();
    int step0 = 1;
    while (2 * step0 < P) step0 *= 2;
    for (int e0 = tid; e0 < n; e0 += U * BLOCK) {
        uint64_t k[U];
        int j[U], a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            k[u] = s_key[min(e0 + u * BLOCK, n - 1)];
            j[u] = a[u] = b[u] = 0;
        }
        for (int step = step0; step > 0; step >>= 1) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int sb = s.begin[min(j[u] + step, P - 1)];
                const uint64_t va = s.v[min(a[u] + step, P - 1) - 1], vb = s.v[min(b[u] + step, P - 1) - 1];
                if (j[u] + step < P && sb <= e0 + u * BLOCK) j[u] += step;
                if (a[u] + step < P && va <= k[u]) a[u] += step;
                if (b[u] + step < P && vb < k[u]) b[u] += step;
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (e0 + u * BLOCK < n) {
                atomicAdd(&s.lt[j[u]][a[u]], 1u);
                atomicAdd(&s.le[j[u]][b[u]], 1u);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int j = q * NW + wave;
        if (j < P) {
            const uint32_t a = incl_scan_u32(s.lt[j][lane]), b = incl_scan_u32(s.le[j][lane]);
            s.lt[j][lane] = a;
            s.le[j][lane] = b;
            if (lane < P - 1) {
                w.myclt[(int64_t)j * P1 + lane + 1] = a;
                w.mycle[(int64_t)j * P1 + lane + 1] = b;
            } else if (lane == P - 1) {
                w.myclt[(int64_t)j * P1] = w.mycle[(int64_t)j * P1] = w.myC[(int64_t)j * P1] = 0;
                w.myclt[(int64_t)j * P1 + P] = w.mycle[(int64_t)j * P1 + P] = sh.begin[j + 1] - sh.begin[j];
            }
        }
    }
    __syncthreads();
    solve_layout<NW>(P, w, sh.C, &s.err, s.c, [&](int r, uint32_t& a, uint32_t& e) {
        const uint32_t cnt = (uint32_t)(sh.begin[lane + 1] - sh.begin[lane]);
        a = r < P - 1 ? s.lt[lane][r] : cnt;
        e = r < P - 1 ? s.le[lane][r] : cnt;
    });
    if (tid < P - 1) {
        w.split[4 * tid] = s.v[tid];
        w.split[4 * tid + 1] = w.split[4 * tid + 2] = w.split[4 * tid + 3] = 0;
    }
}

// key of record i of elsize-byte records with the key at key_off
__device__ __forceinline__ uint64_t byte_key(const uint8_t* sb, int64_t i, int elsize, int key_off, int key_bytes,
                                             const LKey& lk) {
    const uint8_t* p = sb + i * elsize + key_off;
    uint64_t key = 0;
    if (!(((uintptr_t)p | (uintptr_t)key_bytes) & 3) && !(elsize & 3)) {
        const uint32_t* q = reinterpret_cast<const uint32_t*>(p);
        key = q[0];
        if (key_bytes > 4) key |= (uint64_t)q[1] << 32;
    } else {
        for (int b = 0; b < key_bytes; b++) key |= (uint64_t)p[b] << (8 * b);
    }
    return key ^ lk.xmask;
}

// ---------------------------------------------------------------------------
// The smallest sorts: the output position of a record is the number of
// smaller keys plus the equal ones before it, counted outright.  A block
// holds all n <= kRankRecords keys in LDS and places kRankOwn of the records:
// 64 threads per record, each against every 64th key (the reads of a wave
// cover four neighbouring keys, no bank conflict).  n^2 comparisons spread
// over up to 256 workgroups take about 2 us at 4096 records, where the
// dependent steps of a sort inside one workgroup take 38.  The owners of the
// splitters publish them, and the block that finishes last takes the counts
// and the layout from the keys it holds.  in and out must not overlap.
// w.acc: [0] blocks done, [1] [2] the sums; zero between calls.
constexpr int kRankOwn = 16;
template <int RW>
__global__ __launch_bounds__(1024) void rank_sort_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                         LKey lk, int elsize, int key_off, int key_bytes,
                                                         DirectShape sh, DirectWork w, int checksum,
                                                         DirectResult* __restrict__ res) {
    constexpr int BLOCK = 1024, R = kRankOwn, PARTS = BLOCK / R;
    __shared__ uint64_t s_key[kRankRecords];
    __shared__ SmallCounts s_cnt;
    __shared__ uint32_t s_rank[R];
    __shared__ int s_last;
    const int tid = threadIdx.x, lane = tid & 63;
    const int P = sh.P, n = (int)sh.n, i0 = blockIdx.x * R;
    const uint8_t* sb = reinterpret_cast<const uint8_t*>(src);
    long long sum_in = 0, sum_out = 0;
    if (tid < R) s_rank[tid] = 0;
    if (tid == 0) s_cnt.err = 0;
    constexpr int K = kRankRecords / BLOCK;
    if constexpr (RW > 0) {
        uint32_t r[K][RW > 0 ? RW : 1];
#pragma unroll
        for (int k = 0; k < K; k++) RecIO<RW>::load(src, min(k * BLOCK + tid, n - 1), r[k]);
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int i = k * BLOCK + tid;
            s_key[i] = i < n ? lkey<RW>(r[k], lk) : ~0ull;
            if (checksum && i < n && i >= i0 && i < i0 + R) {
#pragma unroll
                for (int q = 0; q < RW; q++) sum_in += sbyte_sum(r[k][q]);
            }
        }
    } else {
        uint64_t v[K];
#pragma unroll
        for (int k = 0; k < K; k++) v[k] = byte_key(sb, min(k * BLOCK + tid, n - 1), elsize, key_off, key_bytes, lk);
#pragma unroll
        for (int k = 0; k < K; k++) s_key[k * BLOCK + tid] = k * BLOCK + tid < n ? v[k] : ~0ull;
    }
    __syncthreads();
    const int own = tid % R, part = tid / R;
    const uint64_t key = s_key[min(i0 + own, n - 1)];
    const int steps = (n + PARTS - 1) / PARTS, s0 = i0 / PARTS;  // the step that holds this block's records
    uint32_t c = 0;
    // padding (the largest key) past n is never counted: equal keys count
    // only before a record
#pragma unroll 8
    for (int s = 0; s < s0; s++) c += s_key[s * PARTS + part] <= key ? 1u : 0u;
    {
        const int i = s0 * PARTS + part;
        const uint64_t k = s_key[i];
        c += k < key || (k == key && i < i0 + own) ? 1u : 0u;
    }
#pragma unroll 8
    for (int s = s0 + 1; s < steps; s++) c += s_key[s * PARTS + part] < key ? 1u : 0u;
    c += __shfl_xor(c, 16, 64);
    c += __shfl_xor(c, 32, 64);
    if (lane < R) atomicAdd(&s_rank[lane], c);
    __syncthreads();
    if constexpr (RW > 0) {
        if (tid < R && i0 + tid < n) {
            uint32_t r[RW > 0 ? RW : 1];
            RecIO<RW>::load(src, i0 + tid, r);
            RecIO<RW>::store(dst, s_rank[tid], r);
            if (checksum) {
#pragma unroll
                for (int q = 0; q < RW; q++) sum_out += sbyte_sum(r[q]);
            }
        }
    } else {
        uint8_t* db = reinterpret_cast<uint8_t*>(dst);
        const int m = min(R, n - i0);
        if (!((elsize | (uintptr_t)sb | (uintptr_t)db) & 3)) {
            const int ew = elsize >> 2;
            for (int x = tid; x < m * ew; x += BLOCK) {
                const int q = x / ew, y = x - q * ew;
                const uint32_t v = src[(int64_t)(i0 + q) * ew + y];
                dst[(int64_t)s_rank[q] * ew + y] = v;
                sum_in += sbyte_sum(v);
                sum_out += sbyte_sum(v);
            }
        } else {
            for (int x = tid; x < m * elsize; x += BLOCK) {
                const int q = x / elsize, y = x - q * elsize;
                const uint8_t v = sb[(int64_t)(i0 + q) * elsize + y];
                db[(int64_t)s_rank[q] * elsize + y] = v;
                sum_in += (signed char)v;
                sum_out += (signed char)v;
            }
        }
    }
    if (checksum) {
        sum_in = wave_sum_ll(sum_in);
        sum_out = wave_sum_ll(sum_out);
        if (lane == 0 && sum_in) atomicAdd(&w.acc[1], (unsigned long long)sum_in);
        if (lane == 0 && sum_out) atomicAdd(&w.acc[2], (unsigned long long)sum_out);
    }
    // splitter i is the key of rank C[i+1] - 1 (0 when C[i+1] is 0)
    for (int x = tid; x < (P - 1) * R; x += BLOCK) {
        const int i = x / R, q = x % R;
        const int64_t Ci = sh.C[i + 1];
        if (i0 + q < n && s_rank[q] == (uint32_t)(Ci > 0 ? Ci - 1 : 0)) store_agent(w.cross + i, s_key[i0 + q]);
    }
    if (tid < R && i0 + tid < n) {
        const uint32_t q = s_rank[tid];
        if (q == 0) w.pminmax[0] = s_key[i0 + tid];
        if (q == (uint32_t)(n - 1)) w.pminmax[4] = s_key[i0 + tid];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0)
        s_last = __hip_atomic_fetch_add(&w.acc[0], 1ull, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) ==
                 (unsigned long long)(gridDim.x - 1);
    __syncthreads();
    if (!s_last) return;
    if (tid < P + 1) w.C[tid] = sh.C[tid];
    if (tid >= 1 && tid < 4) w.pminmax[tid] = w.pminmax[4 + tid] = 0;
    if (P > 1) {
        if (tid < P - 1) s_cnt.v[tid] = load_agent(w.cross + tid);
        __syncthreads();
        small_counts<BLOCK>(sh, w, s_key, s_cnt);
    }
    __syncthreads();
    if (tid < 3) {
        const unsigned long long x = load_agent((uint64_t*)w.acc + tid);
        if (tid) res->sums[tid - 1] = (long long)x;
        store_agent((uint64_t*)w.acc + tid, 0);
        res->lists[tid] = 0;
    }
    if (tid == 3) {
        res->err = s_cnt.err;
        res->scatter_err = 0;
        res->lists[3] = 0;
    }
}

// ---------------------------------------------------------------------------
// Small sorts: at most kSmallRecords records in one workgroup and one launch
// (above kRankRecords, or in place).  The keys stay in LDS; a stable LSD radix
// sort of 16-bit positions over the key bytes that vary (wave-major positions,
// so that equal digits keep their order), the records gathered through the
// cache, then the counts.  Bound by the passes' chains of LDS reads and
// barriers in one workgroup, about 4.8 us a pass at 4096 records (38 of 60 us
// for 8 passes).
// RW = 0: records of elsize bytes with the key at key_off (in and out apart).
constexpr int kSmallWaves = 16, kSmallItems2 = kSmallRecords / (64 * kSmallWaves);
template <int RW>
__global__ __launch_bounds__(1024) void small_sort_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                          LKey lk, int elsize, int key_off, int key_bytes,
                                                          DirectShape sh, DirectWork w, int checksum,
                                                          DirectResult* __restrict__ res) {
    constexpr int BLOCK = 1024, NW = kSmallWaves, K = kSmallItems2;
    __shared__ uint64_t s_key[kSmallRecords];
    __shared__ uint16_t s_idx[2][kSmallRecords];
    __shared__ uint16_t s_whist[NW][kBins];
    __shared__ uint32_t s_excl[kBins];
    __shared__ SmallCounts s_cnt;
    __shared__ uint64_t s_red[2 * NW];
    __shared__ long long s_sum[2][NW];
    __shared__ uint32_t s_tmp[4];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int P = sh.P, n = (int)sh.n;
    const uint8_t* sb = reinterpret_cast<const uint8_t*>(src);
    // keys, their varying bits, and the input sum
    uint64_t any = 0, all = ~0ull;
    long long csum = 0;
    if (tid == 0) s_cnt.err = 0;
    for (int i = tid; i < n; i += BLOCK) {
        uint64_t key;
        if constexpr (RW > 0) {
            uint32_t r[RW > 0 ? RW : 1];
            RecIO<RW>::load(src, i, r);
            key = lkey<RW>(r, lk);
            if (checksum) {
#pragma unroll
                for (int q = 0; q < RW; q++) csum += sbyte_sum(r[q]);
            }
        } else {
            key = byte_key(sb, i, elsize, key_off, key_bytes, lk);
        }
        s_key[i] = key;
        any |= key;
        all &= key;
    }
    if (RW == 0 && checksum)
        for (int64_t b = tid; b < (int64_t)n * elsize; b += BLOCK) csum += (signed char)sb[b];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        any |= __shfl_xor(any, off, 64);
        all &= __shfl_xor(all, off, 64);
    }
    csum = wave_sum_ll(csum);
    if (lane == 0) {
        s_red[wave] = any;
        s_red[NW + wave] = all;
        s_sum[0][wave] = csum;
    }
    __syncthreads();
    any = 0;
    all = ~0ull;
#pragma unroll
    for (int q = 0; q < NW; q++) {
        any |= s_red[q];
        all &= s_red[NW + q];
    }
    const uint64_t vary = any ^ all;
    // the digit passes: wave w owns positions [w span, (w + 1) span)
    const int span = (n + 64 * NW - 1) / (64 * NW) * 64, nk = span / 64;
    const uint64_t lt_mask = __lanemask_lt();
    int cur = 0, passes = 0;
    for (int i = tid; i < n; i += BLOCK) s_idx[0][i] = (uint16_t)i;
    for (int p = 0; p < 8; p++) {
        if (!((vary >> (8 * p)) & 0xffu)) continue;  // uniform
        passes++;
        for (int i = tid; i < NW * kBins / 2; i += BLOCK) reinterpret_cast<uint32_t*>(&s_whist[0][0])[i] = 0;
        __syncthreads();
        volatile uint16_t* wh = s_whist[wave];
        uint32_t dl[K], e[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int pos = wave * span + k * 64 + lane;
            const bool valid = k < nk && pos < n;
            e[k] = valid ? s_idx[cur][pos] : 0u;
            dl[k] = valid ? (uint32_t)(s_key[e[k]] >> (8 * p)) & 0xffu : (uint32_t)kBins;
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (k < nk) {
                const uint32_t d = dl[k];
                const bool valid = d < kBins;
                uint64_t peers = __ballot(valid);
#pragma unroll
                for (int b = 0; b < 8; b++) {
                    const bool bit = (d >> b) & 1u;
                    const uint64_t m = __ballot(bit);
                    peers &= bit ? m : ~m;
                }
                const uint32_t rank = __popcll(peers & lt_mask), cnt = __popcll(peers);
                uint32_t bs = 0;
                if (valid) bs = wh[d];
                dl[k] = d | ((bs + rank) << 16);
                if (valid && rank == 0) wh[d] = (uint16_t)(bs + cnt);
            }
        }
        __syncthreads();
        uint32_t tot = 0;
        if (tid < kBins) {
            uint32_t c[NW];
#pragma unroll
            for (int q = 0; q < NW; q++) c[q] = s_whist[q][tid];
#pragma unroll
            for (int q = 0; q < NW; q++) {
                s_whist[q][tid] = (uint16_t)tot;
                tot += c[q];
            }
        }
        const uint32_t incl = incl_scan_u32(tot);
        if (lane == 63 && wave < 4) s_tmp[wave] = incl;
        __syncthreads();
        if (tid < kBins) {
            uint32_t pre = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) pre += q < wave ? s_tmp[q] : 0u;
            s_excl[tid] = pre + incl - tot;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; k++) {
            const uint32_t d = dl[k] & 0xffffu;
            if (k < nk && d < kBins) s_idx[cur ^ 1][s_excl[d] + s_whist[wave][d] + (dl[k] >> 16)] = (uint16_t)e[k];
        }
        __syncthreads();
        cur ^= 1;
    }
    __syncthreads();
    // every record is read before the first is written (in place)
    csum = 0;
    if constexpr (RW > 0) {
        uint32_t r[K][RW > 0 ? RW : 1];
#pragma unroll
        for (int k = 0; k < K; k++)
            if (k * BLOCK + tid < n) RecIO<RW>::load(src, s_idx[cur][k * BLOCK + tid], r[k]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (k * BLOCK + tid < n) {
                RecIO<RW>::store(dst, k * BLOCK + tid, r[k]);
                if (checksum) {
#pragma unroll
                    for (int q = 0; q < RW; q++) csum += sbyte_sum(r[k][q]);
                }
            }
        }
    } else {
        uint8_t* db = reinterpret_cast<uint8_t*>(dst);
        if (!((elsize | (uintptr_t)sb | (uintptr_t)db) & 3)) {
            const int ew = elsize >> 2;
            for (int64_t x = tid; x < (int64_t)n * ew; x += BLOCK) {
                const int o = (int)(x / ew);
                const uint32_t v = src[(int64_t)s_idx[cur][o] * ew + (x - (int64_t)o * ew)];
                dst[x] = v;
                csum += sbyte_sum(v);
            }
        } else {
            for (int64_t x = tid; x < (int64_t)n * elsize; x += BLOCK) {
                const int o = (int)(x / elsize);
                const uint8_t v = sb[(int64_t)s_idx[cur][o] * elsize + (x - (int64_t)o * elsize)];
                db[x] = v;
                csum += (signed char)v;
            }
        }
    }
    csum = wave_sum_ll(csum);
    if (lane == 0) s_sum[1][wave] = csum;
    if (tid < P + 1) w.C[tid] = sh.C[tid];
    if (P > 1) {
        const uint16_t* si = s_idx[cur];
        if (tid < P - 1) {
            const int Ci = (int)sh.C[tid + 1];
            s_cnt.v[tid] = s_key[si[Ci > 0 ? Ci - 1 : 0]];
        } else if (tid >= BLOCK - 2) {
            const int q = tid - (BLOCK - 2);
            w.pminmax[4 * q] = s_key[si[q ? n - 1 : 0]];
            for (int k = 1; k < 4; k++) w.pminmax[4 * q + k] = 0;
        }
        __syncthreads();
        small_counts<BLOCK>(sh, w, s_key, s_cnt);
    }
    __syncthreads();
    if (tid == 0) {
        long long a = 0, b = 0;
        for (int q = 0; q < NW; q++) {
            a += s_sum[0][q];
            b += s_sum[1][q];
        }
        res->sums[0] = a;
        res->sums[1] = b;
        res->err = s_cnt.err;
        res->scatter_err = 0;
        res->lists[0] = res->lists[1] = res->lists[2] = 0;
        res->lists[3] = (uint32_t)passes;
    }
}

// ---------------------------------------------------------------------------
// host launchers
int launch_direct_sample(int rw, const void* src, const LKey& lk, const DirectShape& sh, const DirectWork& w,
                         bool clear_sums, hipEvent_t start, hipStream_t st) {
    const uint32_t* s = (const uint32_t*)src;
    const unsigned g = (unsigned)std::max(1, sh.S / kDirectChunk);
    switch (rw) {
        case 2: hipExtLaunchKernelGGL(direct_sample_kernel<2>, dim3(g), dim3(kDirectChunk), 0, st, start, nullptr, 0, s, lk, sh, w, clear_sums ? 1 : 0); break;
        case 4: hipExtLaunchKernelGGL(direct_sample_kernel<4>, dim3(g), dim3(kDirectChunk), 0, st, start, nullptr, 0, s, lk, sh, w, clear_sums ? 1 : 0); break;
        default: return -1;
    }
    MPSG_CHECK(hipGetLastError());
    if (g > 1) {
        hipLaunchKernelGGL(direct_rank_kernel, dim3((unsigned)(sh.S / kRankBlock)), dim3(kRankBlock), 0, st, sh.S, sh.W,
                           w.chunks, w.raw);
        MPSG_CHECK(hipGetLastError());
    }
    return 0;
}

int launch_direct_count(int rw, const void* src, const LKey& lk, const DirectShape& sh, const DirectWork& w,
                        long long* checksum, hipStream_t st) {
    const SegDev sd{w.begin, w.count, w.tile_start, sh.P, 0};
    const uint32_t* s = (const uint32_t*)src;
    int step0 = 1;
    while (2 * step0 < sh.W) step0 *= 2;
    const int64_t slots = rw == 2 ? resident_blocks(direct_hist_kernel<2>, 512) : resident_blocks(direct_hist_kernel<4>, 512);
    const int64_t tpb = (sh.ntiles + slots - 1) / slots;
    const unsigned g = (unsigned)((sh.ntiles + tpb - 1) / tpb);
    switch (rw) {
        case 2:
            hipLaunchKernelGGL(direct_hist_kernel<2>, dim3(g), dim3(512), 0, st, s, sd, sh.ntiles, tpb, sh.tile, lk, sh.W,
                               step0, w.raw, w.tables, w.tile_cnt, w.bkt, checksum);
            break;
        case 4:
            hipLaunchKernelGGL(direct_hist_kernel<4>, dim3(g), dim3(512), 0, st, s, sd, sh.ntiles, tpb, sh.tile, lk, sh.W,
                               step0, w.raw, w.tables, w.tile_cnt, w.bkt, checksum);
            break;
        default: return -1;
    }
    MPSG_CHECK(hipGetLastError());
    hipLaunchKernelGGL(direct_scan_kernel, dim3(kLBins / 64), dim3(1024), 0, st, w.tile_cnt, sh.ntiles, w.tile_off, w.tot);
    MPSG_CHECK(hipGetLastError());
    return 0;
}

int launch_direct_counts(int rw, const void* out, const void* part, const LKey& lk, const DirectShape& sh,
                         const DirectWork& w, DirectResult* res, hipEvent_t stop, hipStream_t st) {
    const uint32_t *o = (const uint32_t*)out, *p = (const uint32_t*)part;
    const dim3 g((unsigned)sh.P), b(1024);
    switch (rw) {
        case 2: hipExtLaunchKernelGGL(direct_counts_kernel<2>, g, b, 0, st, nullptr, stop, 0, o, p, lk, sh.P, sh.n, sh.ntiles, w, res); break;
        case 4: hipExtLaunchKernelGGL(direct_counts_kernel<4>, g, b, 0, st, nullptr, stop, 0, o, p, lk, sh.P, sh.n, sh.ntiles, w, res); break;
        default: return -1;
    }
    MPSG_CHECK(hipGetLastError());
    return 0;
}

int launch_small_sort(int rw, const void* src, void* dst, const LKey& lk, int elsize, int key_off, int key_bytes,
                      const DirectShape& sh, const DirectWork& w, bool checksum, bool apart, DirectResult* res,
                      hipEvent_t start, hipEvent_t stop, hipStream_t st) {
    const uint32_t* s = (const uint32_t*)src;
    uint32_t* d = (uint32_t*)dst;
    const int cs = checksum ? 1 : 0;
    const bool by_rank = apart && sh.n <= kRankRecords;
    const dim3 g(by_rank ? (unsigned)((sh.n + kRankOwn - 1) / kRankOwn) : 1u), b(1024);
#define MPSG_SMALL(K, R) \
    hipExtLaunchKernelGGL(K<R>, g, b, 0, st, start, stop, 0, s, d, lk, elsize, key_off, key_bytes, sh, w, cs, res)
    switch (rw + (by_rank ? 16 : 0)) {
        case 0: MPSG_SMALL(small_sort_kernel, 0); break;
        case 1: MPSG_SMALL(small_sort_kernel, 1); break;
        case 2: MPSG_SMALL(small_sort_kernel, 2); break;
        case 4: MPSG_SMALL(small_sort_kernel, 4); break;
        case 8: MPSG_SMALL(small_sort_kernel, 8); break;
        case 16: MPSG_SMALL(rank_sort_kernel, 0); break;
        case 17: MPSG_SMALL(rank_sort_kernel, 1); break;
        case 18: MPSG_SMALL(rank_sort_kernel, 2); break;
        case 20: MPSG_SMALL(rank_sort_kernel, 4); break;
        case 24: MPSG_SMALL(rank_sort_kernel, 8); break;
        default: return -1;
    }
#undef MPSG_SMALL
    MPSG_CHECK(hipGetLastError());
    return 0;
}

}  // namespace mpsg
