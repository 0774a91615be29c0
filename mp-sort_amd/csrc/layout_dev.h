// layout_dev.h -- the layout solve (_solve_for_layout_mpi mpsort-mpi.c:663-727)
// by one workgroup, for the sorts that read their counts off the result.
#pragma once
#include "direct.h"
#include "device.h"

namespace mpsg {

__device__ __forceinline__ uint32_t incl_scan_u32(uint32_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(v, off, 64);
        if (lane >= off) v += o;
    }
    return v;
}

// NW waves; get(r, a, e): CLT and CLE of splitter r in sender `lane` (its size
// for the last receiver); s_c[0] is zero.  Contains one barrier.
template <int NW, class Get>
__device__ __forceinline__ void solve_layout(int P, const DirectWork& w, const int64_t* C, uint32_t* s_err,
                                             uint32_t (*s_c)[kDirectMaxP], Get get) {
    constexpr int Q = kDirectMaxP / NW;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, P1 = P + 1;
    uint32_t a[Q], e[Q];
    int64_t C1[Q], C0[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int r = min(q * NW + wave, P - 1);
        a[q] = e[q] = 0;
        if (lane < P) get(r, a[q], e[q]);
        C0[q] = C[r];
        C1[q] = C[r + 1];
    }
    // counts fit 32 bits: the ranks hold less than 2^31 records together
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int r = q * NW + wave;
        const uint32_t sure = __shfl(incl_scan_u32(a[q]), 63, 64);
        const long long deficit = C1[q] - (long long)sure;
        const uint32_t sp = e[q] > a[q] ? e[q] - a[q] : 0u;
        long long rem = deficit - (long long)(incl_scan_u32(sp) - sp);
        rem = rem > 0 ? rem : 0;
        if (r < P) {
            if (deficit < 0 || (rem > 0 && e[q] < a[q])) atomicOr(s_err, 4u);
            if (lane < P) {
                const uint32_t c = a[q] + (uint32_t)((long long)sp < rem ? (long long)sp : rem);
                s_c[r + 1][lane] = c;
                w.myC[(int64_t)lane * P1 + r + 1] = c;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int r = q * NW + wave;
        if (r < P) {
            const uint32_t x = lane < P ? s_c[r][lane] : 0u, y = lane < P ? s_c[r + 1][lane] : 0u;
            if (y < x) atomicOr(s_err, 8u);
            if (lane < P) w.send[(int64_t)lane * P + r] = (int64_t)y - (int64_t)x;
            const uint32_t sum = incl_scan_u32(y - x);
            if (lane == 63 && (int64_t)sum != C1[q] - C0[q]) atomicOr(s_err, 16u);
        }
    }
}

}  // namespace mpsg
