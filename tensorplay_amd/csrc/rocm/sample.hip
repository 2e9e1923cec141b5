// Top-k / top-p draws with k > 1024 (k = cols: top-p alone) without sorting the
// row: one workgroup per row finds the nucleus end and the drawn position by
// weight.  The draw's definition is tpr_sample's (tpr_rocm.h): in the order of
// tpr_topk (key descending, lowest index first), with w_j = exp((v_j - v_0)/T)
// and c_j = w_0 + .. + w_j, m is the first j with c_j >= top_p * c_{k-1} and
// the answer the first j <= m with c_j > u * c_m.
//
// k_sample_row, in phases:
//   1. The row is read from HBM once: VR float4 per thread stay in registers,
//      what is left over streams (and is read again from the caches in phase 2).
//      The row's maximum v_0 comes from the same pass.
//   2. c_{k-1} (float64 sums) and a candidate list.  No more than k elements lie
//      below v_0 - T * ln(k / (1 - top_p)), each with a weight under (1 - top_p)
//      / k, so together they weigh less than (1 - top_p) * w_0 <= (1 - top_p) *
//      c_{k-1}: the nucleus ends among the elements at or above that bound, and
//      only those are listed and sorted.  The list is also kept short: a second
//      bound is the largest over the waves of the least thread maximum, which
//      about 512 * ln 64 elements of a row in random order reach (2100 of 151936
//      logits); it promises nothing, but phase 3 sees whether it held.
//   3. The sorted list's prefix sums (float64) give m and the draw, if they
//      reach the nucleus end.
// top_p = 1, and rows whose list overflows or ends before the nucleus does (flat
// distributions), take draw_by_radix: the position where the weight from the top reaches a target is
// found by three radix passes over the keys (11 / 11 / 10 bits) with a
// histogram of 64-bit fixed-point weights in LDS -- integer sums, so the
// result does not depend on the order of the additions -- once for m and once
// for the draw.  k < cols first finds the k-th key the same way with every
// weight 1.  Rows whose largest element is NaN or infinite have no finite c_j:
// the definition then leaves position k - 1.
//
// What bounds it: the one read of the row, then the exponentials (12
// instructions an element) and the fixed tail (sort, scans).  512 threads, so
// that a thread may hold 216 of a row's values (54 float4, 252 registers).
// MI355X, k = cols, against the sort of all candidates in the workspace that
// this replaced: [256, 151936] T 0.8 top_p 0.9 6070 -> 80 us, [256, 50257] 1075
// -> 42, [1, 151936] 3976 -> 50; the radix draws (T 1, top_p 1) 275 / 92 / 153.
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "common.h"
#include "sample.h"
#include "select.h"

namespace tpr {
namespace {

constexpr int kNT = 512;      // threads per row
constexpr int kNW = kNT / 64;
constexpr int kList = 4096;   // candidates sorted in phase 3 (8 per thread)
constexpr int kListK = 1600;  // largest k tried on a list cut by the bound of phase 2
constexpr int kBins = 2048;
constexpr int kUnitRow = 1 << 20;  // rows from here on: draw_by_radix's unit comes from the row's total

typedef float f4 __attribute__((ext_vector_type(4)));
typedef f4 f4u __attribute__((aligned(4)));  // rows start at any element
typedef unsigned long long u64;

struct SampleArgs {
    const float* in;
    int cols;
    long long row_stride;
    int k;
    float temperature, top_p;
    float scale;       // fixed-point weight of the largest element of a row shorter than kUnitRow (a power of two)
    float c_hi, c_lo;  // log2(e) / temperature as a float pair
    float span;        // temperature * ln(k / (1 - top_p)); < 0: no list
    const float* u;
    long long* ids;
};

struct SampleShared {
    union {
        u64 list[kList];
        u64 hist0[kBins];  // draw_by_radix: the first digit's weights
    };
    union {
        u64 hist[kBins];
        u64 xb[kNT * 4];  // reg_sort_desc's exchanges
    };
    double dsum[kNW];
    u64 wsum[kNW];
    float fmax_[kNW], fmin_[kNW];
    int nan_[kNW];
    int wmin[2][kNW];
    int count;
    int digit;
    u64 above;
    double cm;
};

// exp((v - v0) / T) for d = v - v0 <= 0: the exponent in base 2 as a float pair,
// so the product's rounding does not enter the weight.  0 below 2^-126 (and for
// v = -inf).
__device__ __forceinline__ float weight(float d, const SampleArgs& a) {
    const float q = d * a.c_hi;
    const float lo = fmaf(d, a.c_lo, fmaf(d, a.c_hi, -q));
    const float e = __builtin_amdgcn_exp2f(q);
    const float w = fmaf(e, lo * 0.693147181f, e);
    return q > -126.0f ? w : 0.0f;
}

// f(value, index) for the elements [first, n) of the row, strided over the
// workgroup, four vectors in flight per thread.
template <class F>
__device__ __forceinline__ void stream_row(const float* p, int first, int n, F&& f) {
    const int nv = n >> 2;
    int i = (first >> 2) + threadIdx.x;
    for (; i + 3 * kNT < nv; i += 4 * kNT) {
        f4 v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = *reinterpret_cast<const f4u*>(p + 4ll * (i + q * kNT));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int c = 0; c < 4; ++c) f(v[q][c], 4 * (i + q * kNT) + c);
        }
    }
    for (; i < nv; i += kNT) {
        const f4 v = *reinterpret_cast<const f4u*>(p + 4ll * i);
#pragma unroll
        for (int c = 0; c < 4; ++c) f(v[c], 4 * i + c);
    }
    const unsigned t = (unsigned)(nv << 2) + threadIdx.x;  // may pass 2^31
    if (t < (unsigned)n) f(p[t], (int)t);
}

__device__ double block_sum(double v, double* sh) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) v += __shfl_xor(v, m, 64);
    __syncthreads();
    if (__lane_id() == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = 0.0;
#pragma unroll
    for (int i = 0; i < kNW; ++i) r += sh[i];
    return r;
}

__device__ int block_min(int v, int* sh) {
    v = __ockl_wfred_min_i32(v);
    if (__lane_id() == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    int r = sh[0];
#pragma unroll
    for (int i = 1; i < kNW; ++i) r = min(r, sh[i]);
    return r;
}

// The digit of a 2048-bin histogram (counted from the top bin) in which the
// running weight from the top, starting at `above`, reaches `target`:
// sh.digit, and sh.above = the weight above that bin.  target <= above + total.
__device__ void find_digit(SampleShared& sh, const u64* hist, u64 above, u64 target) {
    constexpr int BPT = kBins / kNT;
    const int t = threadIdx.x, lane = __lane_id(), w = t >> 6;
    const int rt = kNT - 1 - t;  // thread 0 owns the highest bins
    u64 h[BPT], own = 0;
#pragma unroll
    for (int b = 0; b < BPT; ++b) {
        h[b] = hist[rt * BPT + b];
        own += h[b];
    }
    u64 incl = own;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        const u64 x = __shfl_up(incl, m, 64);
        if (lane >= m) incl += x;
    }
    if (lane == 63) sh.wsum[w] = incl;
    __syncthreads();
    u64 before = above;
#pragma unroll
    for (int i = 0; i < kNW; ++i)
        if (i < w) before += sh.wsum[i];
    incl += before;
    const u64 excl = incl - own;
    if (incl >= target && excl < target) {  // one thread
        u64 c = excl;
        int b = BPT - 1;
        for (; b > 0; --b) {
            if (c + h[b] >= target) break;
            c += h[b];
        }
        sh.digit = rt * BPT + b;
        sh.above = c;
    }
    __syncthreads();
}

// The fixed-point weight of an element, in units of 1 / scale; unit: every
// element weighs 1.
__device__ __forceinline__ u64 fixed_weight(float v, float v0, bool unit, float scale, const SampleArgs& a) {
    return unit ? 1ull : (u64)(weight(v - v0, a) * scale);
}

struct Pick {
    uint32_t key;  // the position's key
    u64 above;     // weight of every element with a larger key
};

__device__ void first_digit_hist(SampleShared& sh, u64* hist, const float* p, int n, float v0, bool unit,
                                 float scale, const SampleArgs& a) {
    for (int i = threadIdx.x; i < kBins; i += kNT) hist[i] = 0;
    __syncthreads();
    stream_row(p, 0, n, [&](float v, int) {
        const u64 w = fixed_weight(v, v0, unit, scale, a);
        if (w) atomicAdd(&hist[f2key(v, 1) >> 21], w);
    });
    __syncthreads();
}

// The key of the first position whose running weight reaches `target` (1 <=
// target <= the total weight in hist0, the first digit's histogram).
__device__ Pick pick(SampleShared& sh, const u64* hist0, const float* p, int n, float v0, bool unit, float scale,
                     u64 target, const SampleArgs& a) {
    find_digit(sh, hist0, 0, target);
    uint32_t prefix = (uint32_t)sh.digit << 21;
    u64 above = sh.above;
    for (int level = 1; level < 3; ++level) {
        const int shift = level == 1 ? 10 : 0;
        const uint32_t pmask = level == 1 ? 0xffe00000u : 0xfffffc00u;
        const uint32_t dmask = level == 1 ? 0x7ffu : 0x3ffu;
        __syncthreads();
        for (int i = threadIdx.x; i < kBins; i += kNT) sh.hist[i] = 0;
        __syncthreads();
        stream_row(p, 0, n, [&](float v, int) {
            const uint32_t key = f2key(v, 1);
            if ((key & pmask) == prefix) {
                const u64 w = fixed_weight(v, v0, unit, scale, a);
                if (w) atomicAdd(&sh.hist[(key >> shift) & dmask], w);
            }
        });
        __syncthreads();
        find_digit(sh, sh.hist, above, target);
        prefix |= (uint32_t)sh.digit << shift;
        above = sh.above;
    }
    __syncthreads();
    return {prefix, above};
}

// Index of the ord-th (from 1) element, in index order, whose key is `key`;
// every wave counts a contiguous piece of the row, then the wave that holds
// the element scans its piece.
__device__ void locate(SampleShared& sh, const float* p, int n, uint32_t key, u64 ord, long long* out) {
    const int lane = __lane_id(), w = threadIdx.x >> 6;
    const long long piece = (((long long)n + kNW - 1) / kNW + 63) & ~63ll;
    // unsigned: a step past hi may pass 2^31
    const unsigned lo = (unsigned)min((long long)n, w * piece), hi = (unsigned)min((long long)n, (w + 1) * piece);
    u64 cnt = 0;
    unsigned b = lo;
    for (; b + 512 <= hi; b += 512) {
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = (p + b)[q * 64 + lane];
#pragma unroll
        for (int q = 0; q < 8; ++q) cnt += (u64)__popcll(__ballot(f2key(v[q], 1) == key));
    }
    for (; b < hi; b += 64) cnt += (u64)__popcll(__ballot(b + lane < hi && f2key(p[min(b + lane, hi - 1)], 1) == key));
    __syncthreads();
    if (lane == 0) sh.wsum[w] = cnt;
    __syncthreads();
    u64 before = 0;
#pragma unroll
    for (int i = 0; i < kNW; ++i)
        if (i < w) before += sh.wsum[i];
    if (before < ord && before + cnt >= ord) {
        for (b = lo; b < hi; b += 64) {
            const bool hit = b + lane < hi && f2key(p[min(b + lane, hi - 1)], 1) == key;
            const u64 bal = __ballot(hit);
            const u64 c = (u64)__popcll(bal);
            if (before + c >= ord) {
                if (hit && before + (u64)__popcll(bal & lanemask_lt()) + 1 == ord) *out = b + lane;
                break;
            }
            before += c;
        }
    }
}

// Position `target` - 1 in rank order (every element weighs 1).
__device__ Pick pick_rank(SampleShared& sh, const float* p, int n, u64 target, const SampleArgs& a) {
    first_digit_hist(sh, sh.hist, p, n, 0.0f, true, 0.0f, a);
    const Pick r = pick(sh, sh.hist, p, n, 0.0f, true, 0.0f, target, a);
    return r;
}

// The top k's float64 weight that lies on the kties elements of the k-th key.
__device__ __forceinline__ double ties_weight(float v0, uint32_t kth, u64 kties, const SampleArgs& a) {
    return kties ? (double)kties * (double)weight(__uint_as_float(key2bits(kth, 1)) - v0, a) : 0.0;
}

// m and the draw by weighted radix selection over the row in memory.  kth /
// kties: the k-th key and how many of its elements are among the top k.  total:
// the top k's float64 weight, below 0 if the caller has not formed it.
//
// The unit of the fixed-point weights: an element loses less than one unit to
// it, a row less than n units.  Rows of fewer than kUnitRow elements leave room
// for n weights of 1 (a.scale; at most 2^44): a loss below 2^-22 of v_0's weight
// alone, less than the float32 sums of a sorted row lose.  Longer rows would lose
// more (2^24 elements: 2^-13 of v_0's weight) and take the unit from their total,
// which then fills 62 bits: n units are less than 2^(31 - 61) of it.  Where the
// total has not been formed (top_p = 1) that is one more pass.  LONG is a template
// parameter: as a test here it cost rows of 10^6 3%.
template <bool LONG>
__device__ void draw_by_radix(SampleShared& sh, const float* p, int n, float v0, uint32_t kth, u64 kties, float u,
                              double total_w, const SampleArgs& a, long long* out) {
    float scale = a.scale;
    if constexpr (LONG) {
        if (total_w < 0.0) {
            double s = 0.0;
            stream_row(p, 0, n, [&](float v, int) {
                if (f2key(v, 1) > kth) s += (double)weight(v - v0, a);
            });
            total_w = block_sum(s, sh.dsum) + ties_weight(v0, kth, kties, a);
        }
        // 1 <= total_w < 2^31: the weights' sum stays below 2^62
        scale = ldexpf(1.0f, 61 - __builtin_amdgcn_readfirstlane(ilogb(total_w)));
    }
    // the top k's weights by first digit, and their sum
    for (int i = threadIdx.x; i < kBins; i += kNT) sh.hist0[i] = 0;
    __syncthreads();
    stream_row(p, 0, n, [&](float v, int) {
        const uint32_t key = f2key(v, 1);
        if (key > kth) {
            const u64 w = fixed_weight(v, v0, false, scale, a);
            if (w) atomicAdd(&sh.hist0[key >> 21], w);
        }
    });
    if (kties && threadIdx.x == 0) {
        const u64 w = fixed_weight(__uint_as_float(key2bits(kth, 1)), v0, false, scale, a);
        if (w) atomicAdd(&sh.hist0[kth >> 21], w * kties);
    }
    __syncthreads();
    u64 s = 0;
#pragma unroll
    for (int b = 0; b < kBins / kNT; ++b) s += sh.hist0[b * kNT + threadIdx.x];
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) s += __shfl_xor(s, m, 64);
    if (__lane_id() == 0) sh.wsum[threadIdx.x >> 6] = s;
    __syncthreads();
    u64 total = 0;
#pragma unroll
    for (int i = 0; i < kNW; ++i) total += sh.wsum[i];
    __syncthreads();
    const double cut = ceil((double)a.top_p * (double)total);
    const u64 t1 = a.top_p >= 1.0f ? total : min(total, max((u64)1, (u64)cut));
    const Pick m = pick(sh, sh.hist0, p, n, v0, false, scale, t1, a);
    const u64 wm = fixed_weight(__uint_as_float(key2bits(m.key, 1)), v0, false, scale, a);
    const u64 ties = (t1 - m.above + wm - 1) / wm;
    const u64 cm = m.above + ties * wm;
    const double thr = (double)u * (double)cm;
    // the first c_j > thr; u >= 1 or NaN leaves m
    const u64 t2 = thr < (double)cm ? (thr < 0.0 ? 1ull : min(cm, (u64)thr + 1ull)) : cm;
    const Pick d = pick(sh, sh.hist0, p, n, v0, false, scale, t2, a);
    const u64 wd = fixed_weight(__uint_as_float(key2bits(d.key, 1)), v0, false, scale, a);
    locate(sh, p, n, d.key, (t2 - d.above + wd - 1) / wd, out);
}

// m and the draw from the sorted list; false if the list does not reach the
// nucleus end.  A negative total: the list holds the top k, whose weight is the
// list's own.
__device__ bool draw_from_list(SampleShared& sh, int cnt, int k, float v0, double total, float u, const SampleArgs& a,
                               long long* out) {
    constexpr int P = kList / kNT;
    const int t = threadIdx.x, lane = __lane_id(), w = t >> 6;
    int n2 = 64 * P;
    while (n2 < cnt) n2 <<= 1;
    u64 x[P];
#pragma unroll
    for (int q = 0; q < P; ++q) x[q] = (t * P + q < cnt) ? sh.list[t * P + q] : 0ull;
    reg_sort_desc<kNT, P>(x, sh.xb, n2);
    const int last = min(cnt, k) - 1;
    double pw[P], s = 0.0;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        const int j = t * P + q;
        pw[q] = j <= last ? (double)weight(__uint_as_float(key2bits((uint32_t)(x[q] >> 32), 1)) - v0, a) : 0.0;
        s += pw[q];
    }
    double incl = s;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        const double y = __shfl_up(incl, m, 64);
        if (lane >= m) incl += y;
    }
    if (lane == 63) sh.dsum[w] = incl;
    __syncthreads();
    double before = 0.0;
#pragma unroll
    for (int i = 0; i < kNW; ++i)
        if (i < w) before += sh.dsum[i];
    const double excl = before + (incl - s);
    const bool whole = total < 0.0;
    if (whole) {
        total = 0.0;
#pragma unroll
        for (int i = 0; i < kNW; ++i) total += sh.dsum[i];
    }
    const double cut = (double)a.top_p * total;
    int mj = 0x7fffffff;
    double c = excl;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        c += pw[q];
        if (c >= cut && mj == 0x7fffffff && t * P + q <= last) mj = t * P + q;
    }
    int m = block_min(mj, sh.wmin[0]);
    if (m > last) {
        if (!whole) return false;
        m = last;  // c_{k-1} reaches the cut whatever the roundings
    }
    c = excl;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        c += pw[q];
        if (t * P + q == m) sh.cm = c;
    }
    __syncthreads();
    const double thr = (double)u * sh.cm;
    int dj = 0x7fffffff;
    c = excl;
#pragma unroll
    for (int q = 0; q < P; ++q) {
        c += pw[q];
        if (c > thr && dj == 0x7fffffff && t * P + q <= m) dj = t * P + q;
    }
    const int d = min(block_min(dj, sh.wmin[1]), m);
#pragma unroll
    for (int q = 0; q < P; ++q)
        if (t * P + q == d) *out = (long long)comp_index(x[q]);
    return true;
}

// VR float4 of the row per thread in registers (the host picks VR with VR * 4 *
// kNT <= cols, so the register part needs no range checks).  ALL: k = cols (no
// k-th key; the test per element on it costs registers and time).  LONG: rows of
// kUnitRow elements or more.
template <int VR, bool ALL, bool LONG = false>
__global__ __launch_bounds__(kNT) void k_sample_row(SampleArgs a) {
    __shared__ SampleShared sh;
    const long long row = blockIdx.x;
    const float* p = a.in + row * a.row_stride;
    const int n = a.cols, t = threadIdx.x;
    constexpr int kReg = VR * kNT * 4;  // elements held
    f4 x[VR ? VR : 1];
#pragma unroll
    for (int j = 0; j < VR; ++j)
        x[j] = __builtin_nontemporal_load(reinterpret_cast<const f4u*>(p + 4 * (j * kNT + t)));
    if (t == 0) sh.count = 0;
    // 1. the maximum; NaN counts as larger than everything
    float mx = -INFINITY;
    int nan = 0;
    auto top = [&](float v, int) {
        mx = fmaxf(mx, v);
        nan |= v != v;
    };
    stream_row(p, kReg, n, top);
#pragma unroll
    for (int j = 0; j < VR; ++j) {
#pragma unroll
        for (int c = 0; c < 4; ++c) top(x[j][c], 0);
    }
    float lo = mx;  // least of the wave's thread maxima
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        mx = fmaxf(mx, xor_lane_f(mx, m));
        lo = fminf(lo, xor_lane_f(lo, m));
    }
    nan = __any(nan) ? 1 : 0;
    if (__lane_id() == 0) {
        sh.fmax_[t >> 6] = mx;
        sh.fmin_[t >> 6] = lo;
        sh.nan_[t >> 6] = nan;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kNW; ++i) {
        mx = fmaxf(mx, sh.fmax_[i]);
        nan |= sh.nan_[i];
        lo = fmaxf(lo, sh.fmin_[i]);
    }
    const float v0 = mx;
    const uint32_t key0 = nan ? f2key(NAN, 1) : f2key(v0, 1);
    if (!(a.temperature > 0.0f)) {  // greedy
        locate(sh, p, n, key0, 1, &a.ids[row]);
        return;
    }
    if (nan || v0 == INFINITY || v0 == -INFINITY) {  // no finite sums: position k - 1
        const Pick r = pick_rank(sh, p, n, (u64)a.k, a);
        locate(sh, p, n, r.key, (u64)a.k - r.above, &a.ids[row]);
        return;
    }
    const float u = a.u[row];
    uint32_t kth = 0;  // every element is above key 0
    u64 kties = 0;
    if constexpr (!ALL) {
        // Small k: the bound that keeps the list short (phase 2) often leaves the
        // whole top k on it -- about 1700 elements reach it -- and the sorted list
        // then is the answer, where the k-th key costs three more passes
        // ([64, 16000] k = 1050 48 -> 36 us, [64, 151936] 141 ->
        // 101).  Rows of kList or less would sort all of themselves ([64, 2097]
        // 33 against 25).
        if (n > kList && a.k <= kListK) {
            stream_row(p, 0, n, [&](float v, int i) {
                if (v >= lo) {
                    const int at = atomicAdd(&sh.count, 1);
                    if (at < kList) sh.list[at] = comp_key(f2key(v, 1), (uint32_t)i);
                }
            });
            __syncthreads();
            const int cnt = sh.count;
            __syncthreads();
            if (cnt >= a.k && cnt <= kList) {
                draw_from_list(sh, cnt, a.k, v0, -1.0, u, a, &a.ids[row]);
                return;
            }
            if (t == 0) sh.count = 0;
            __syncthreads();
        }
        const Pick r = pick_rank(sh, p, n, (u64)a.k, a);
        kth = r.key;
        kties = (u64)a.k - r.above;
    }
    double total = -1.0;
    if (a.span >= 0.0f) {
        // 2. the top k's total weight and the elements at or above the bound
        float bound = v0 - a.span;
        bound -= fabsf(bound) * 2.4e-7f;  // never above the exact difference
        if (n > kList) bound = fmaxf(bound, lo);
        double tot = 0.0;
        // a vector's weights (summed in float32, then added in float64); true
        // if one of its elements belongs on the list
        auto add = [&](f4 v) {
            float s = 0.0f;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (ALL || f2key(v[c], 1) > kth) s += weight(v[c] - v0, a);
            tot += (double)s;
            return fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])) >= bound;
        };
        auto list = [&](float v, int i) {
            const uint32_t key = f2key(v, 1);
            if (v >= bound && key >= kth) {
                const int at = atomicAdd(&sh.count, 1);
                if (at < kList) sh.list[at] = comp_key(key, (uint32_t)i);
            }
        };
        u64 hits = 0;
#pragma unroll
        for (int j = 0; j < VR; ++j) hits |= add(x[j]) ? 1ull << j : 0ull;
        // few: read again, four at a time, rather than indexed in the registers
        while (hits) {
            int i[4];
            f4 v[4];
            const int first = __ffsll(hits) - 1;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = hits ? __ffsll(hits) - 1 : -1;
                hits &= hits - 1;
                i[q] = j < 0 ? -1 : 4 * (j * kNT + t);
                v[q] = *reinterpret_cast<const f4u*>(p + 4 * ((j < 0 ? first : j) * kNT + t));
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (i[q] >= 0)
                    for (int c = 0; c < 4; ++c) list(v[q][c], i[q] + c);
        }
        const int nv = n >> 2;
        int i = VR * kNT + t;
        for (; i + 7 * kNT < nv; i += 8 * kNT) {  // eight vectors in flight
            f4 v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = *reinterpret_cast<const f4u*>(p + 4ll * (i + q * kNT));
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (add(v[q]))
                    for (int c = 0; c < 4; ++c) list(v[q][c], 4 * (i + q * kNT) + c);
        }
        for (; i < nv; i += kNT) {
            const f4 v = *reinterpret_cast<const f4u*>(p + 4ll * i);
            if (add(v))
                for (int c = 0; c < 4; ++c) list(v[c], 4 * i + c);
        }
        const unsigned e = (unsigned)(nv << 2) + threadIdx.x;  // may pass 2^31
        if (e < (unsigned)n) {
            const float v = p[e];
            if (ALL || f2key(v, 1) > kth) tot += (double)weight(v - v0, a);
            list(v, (int)e);
        }
        total = block_sum(tot, sh.dsum);
        total += ties_weight(v0, kth, kties, a);
        const int cnt = sh.count;
        __syncthreads();
        if (cnt <= kList) {
            if (draw_from_list(sh, cnt, a.k, v0, total, u, a, &a.ids[row])) return;
            __syncthreads();
        }
    }
    draw_by_radix<LONG>(sh, p, n, v0, kth, kties, u, total, a, &a.ids[row]);
}

}  // namespace

int sample_rows(const float* in, long long rows, long long cols, long long row_stride, long long k, float temperature,
                float top_p, const float* u, long long* ids, hipStream_t st) {
    const long long most = kMaxThreads / kNT;  // rows of one launch
    if (rows > most) {
        const int rc = sample_rows(in, most, cols, row_stride, k, temperature, top_p, u, ids, st);
        if (rc != TPR_OK) return rc;
        return sample_rows(in + most * row_stride, rows - most, cols, row_stride, k, temperature, top_p, u + most,
                           ids + most, st);
    }
    SampleArgs a;
    a.in = in;
    a.cols = (int)cols;
    a.row_stride = row_stride;
    a.k = (int)k;
    a.temperature = temperature;
    a.top_p = top_p;
    const double c = temperature > 0.0f ? std::fmin(1.4426950408889634074 / (double)temperature, 3.4e38) : 0.0;
    a.c_hi = (float)c;
    a.c_lo = std::isfinite(a.c_hi) ? (float)(c - (double)a.c_hi) : 0.0f;
    // one ulp of room for the roundings of the bound and of the weights
    const double span = (double)temperature * (std::log((double)k / (1.0 - (double)top_p)) * 1.0001 + 1e-4);
    a.span = (top_p < 1.0f && temperature > 0.0f && std::isfinite(span) && span < 3e38) ? (float)span : -1.0f;
    int sh = 62;
    while (sh > 0 && (cols >> (62 - sh)) > 0) --sh;  // cols * 2^sh < 2^62
    a.scale = std::ldexp(1.0f, sh < 44 ? sh : 44);
    a.u = u;
    a.ids = ids;
    const dim3 g((unsigned)rows), b(kNT);
    const long long per = cols / (4 * kNT);  // whole vectors per thread
#define TPR_SAMPLE(...) hipLaunchKernelGGL((k_sample_row<__VA_ARGS__>), g, b, 0, st, a)
    if (cols >= kUnitRow) {
        if (k < cols) TPR_SAMPLE(0, false, true);
        else TPR_SAMPLE(54, true, true);
    } else if (k < cols) TPR_SAMPLE(0, false);
    else if (per >= 54) TPR_SAMPLE(54, true);
    else if (per >= 36) TPR_SAMPLE(36, true);
    else if (per >= 24) TPR_SAMPLE(24, true);
    else if (per >= 14) TPR_SAMPLE(14, true);
    else if (per >= 6) TPR_SAMPLE(6, true);
    else TPR_SAMPLE(0, true);
#undef TPR_SAMPLE
    return check_launch("k_sample_row");
}

}  // namespace tpr
