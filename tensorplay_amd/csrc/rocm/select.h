// Sortable keys, composites and the register bitonic sort shared by the top-k
// and sampling kernels.
#pragma once

#include "common.h"

namespace tpr {

// Order-preserving float -> uint32 map: non-negative u -> u | 2^31, negative
// u -> ~u + 1 (two's-complement negate of the magnitude's image), so -0.0 and
// +0.0 land on the same key 2^31; every NaN is first made 0x7fc00000 (above
// +inf).  lmask = 0 keeps the order (largest), ~0 reverses it (smallest).
// Valid keys are never 0: 0 marks "no element".  Branch-free: one NaN compare
// (f != f) and select, an arithmetic shift, xor, subtract, xor.
__device__ __forceinline__ uint32_t f2key_sel(float f, uint32_t lmask) {
    const uint32_t u = (f != f) ? 0x7fc00000u : __float_as_uint(f);
    const uint32_t m = (uint32_t)((int32_t)u >> 31);
    return ((u ^ (m | 0x80000000u)) - m) ^ lmask;
}

__device__ __forceinline__ uint32_t f2key(float f, int largest) {
    return f2key_sel(f, largest ? 0u : 0xffffffffu);
}

// Inverse of f2key.  Exact except for the two canonicalised cases (-0.0 comes
// back as +0.0, any NaN as 0x7fc00000); callers re-read the input for those.
__device__ __forceinline__ uint32_t key2bits(uint32_t key, int largest) {
    const uint32_t k = largest ? key : ~key;
    return (k & 0x80000000u) ? (k & 0x7fffffffu) : (0u - k);
}

__device__ __forceinline__ unsigned long long comp_key(uint32_t key, uint32_t idx) {
    return ((unsigned long long)key << 32) | (unsigned long long)(0xffffffffu - idx);
}

__device__ __forceinline__ uint32_t comp_index(unsigned long long c) {
    return 0xffffffffu - (uint32_t)(c & 0xffffffffull);
}

// Inclusive prefix sum over the wave's 64 lanes (every lane active): DPP row
// shifts by 1, 2, 4, 8 (lanes whose source is outside the row add the 0 passed
// as `old`), then row_bcast:15 and row_bcast:31 carry the row totals upward.
// No LDS round trips.
__device__ __forceinline__ int wave_incl_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}

__device__ __forceinline__ unsigned long long lanemask_lt() { return (1ull << __lane_id()) - 1ull; }

template <int M, int P>
__device__ __forceinline__ void sort_lane_stage(unsigned long long (&x)[P], bool keep_max) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const uint32_t lo = xor_lane<M>((uint32_t)x[p]);
        const uint32_t hi = xor_lane<M>((uint32_t)(x[p] >> 32));
        const unsigned long long y = ((unsigned long long)hi << 32) | lo;
        x[p] = ((x[p] > y) == keep_max) ? x[p] : y;
    }
}

// Descending bitonic sort of n composites (n / P threads, a multiple of 64,
// at most NT) held P per thread: thread t holds positions t*P .. t*P+P-1.
// Distances below P: compare-exchanges in registers; below 64*P: the partner
// lane's value by a lane permute; the rest through xb (LDS, NT*min(P, 4)
// composites) with a barrier, which every thread of the workgroup reaches.
template <int NT, int P>
__device__ void reg_sort_desc(unsigned long long (&x)[P], unsigned long long* xb, int n) {
    constexpr int Q = P < 4 ? P : 4;
    const int t = threadIdx.x;
    const bool active = t < n / P;  // whole waves
    for (int s = 2; s <= n; s <<= 1) {
        for (int d = s >> 1; d >= P; d >>= 1) {
            const int m = d / P;  // partner thread t ^ m
            const bool desc = ((t * P) & s) == 0;
            const bool keep_max = ((t & m) == 0) == desc;
            if (!active && m < 64) continue;
            switch (m) {
                case 1: sort_lane_stage<1, P>(x, keep_max); break;
                case 2: sort_lane_stage<2, P>(x, keep_max); break;
                case 4: sort_lane_stage<4, P>(x, keep_max); break;
                case 8: sort_lane_stage<8, P>(x, keep_max); break;
                case 16: sort_lane_stage<16, P>(x, keep_max); break;
                case 32: sort_lane_stage<32, P>(x, keep_max); break;
                default:
#pragma unroll
                    for (int p0 = 0; p0 < P; p0 += Q) {
                        if (active) {
#pragma unroll
                            for (int q = 0; q < Q; ++q) xb[q * NT + t] = x[p0 + q];
                        }
                        __syncthreads();
                        if (active) {
#pragma unroll
                            for (int q = 0; q < Q; ++q) {
                                const unsigned long long y = xb[q * NT + (t ^ m)];
                                x[p0 + q] = ((x[p0 + q] > y) == keep_max) ? x[p0 + q] : y;
                            }
                        }
                        __syncthreads();
                    }
            }
        }
        if (!active) continue;
#pragma unroll
        for (int dd = P / 2; dd >= 1; dd >>= 1) {
            if (dd < s) {
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    if ((p & dd) == 0) {
                        const bool desc = ((t * P + p) & s) == 0;
                        const unsigned long long u = x[p], v = x[p + dd];
                        const bool sw = (u > v) != desc;
                        x[p] = sw ? v : u;
                        x[p + dd] = sw ? u : v;
                    }
                }
            }
        }
    }
}

}  // namespace tpr
