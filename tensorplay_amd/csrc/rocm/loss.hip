// gfx950 nll_loss forward and backward, behind tpr_nll_loss() and
// tpr_nll_loss_backward().
//
// Forward follows the CPU kernel
// (/root/reference/p10/src/backend/cpu/LossKernels.cpp:12-55):
//   loss_i = -x[i, t_i] * w[t_i] (float32), 0 for ignored samples;
//   total_weight = sum of w[t_i] over samples that are not ignored;
//   mean = sum(loss_i) / total_weight when total_weight > 0, sum = sum(loss_i).
// The reference sums the losses in double (as here) and the weights in float
// sequentially (here in double, then rounded once to float: identical for
// unit weights, and within one rounding otherwise).  The CUDA path
// (LossKernels.cu:38-61) instead does float atomicAdds, whose order varies run
// to run; here partial sums per workgroup are combined in a fixed order by a
// second one-workgroup kernel, so results are deterministic.
// Backward writes grad_input in one pass (zeros plus the target element),
// instead of the reference's zeros() then scatter.

#include <hip/hip_runtime.h>

#include <string>

#include "common.h"
#include "nll_walk.h"

namespace tpr {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef f32x4_t f32x4_any __attribute__((aligned(4)));  // outputs start at any float

constexpr int kNllBlock = 256;
constexpr int kNllMaxBlocks = 1024;
constexpr long long kNllOne = 4096;  // most samples of the single-workgroup forward

struct NllPart {
    double loss;
    double weight;
    int bad;
    int pad;
};

struct NllArgs {
    const float* x;
    long long n, c, s0, s1;
    const long long* t;
    long long ts;
    const float* w;
    long long reduction, ignore;
    float* out;       // [n] for reduction none
    NllPart* part;    // one per workgroup
};

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int o = kWave / 2; o >= 1; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

struct NllFin {
    const NllPart* part;
    int nparts;
    long long reduction;
    float* out;
    float* total_weight;
    int* status;
};

__device__ __forceinline__ void nll_finish(const NllFin& f, const NllPart& p) {
    double l = p.loss;
    const float tw = (float)p.weight;
    if (f.reduction == 1 && tw > 0.0f) l /= (double)tw;
    if (f.reduction != 0) f.out[0] = (float)l;
    f.total_weight[0] = tw;
    if (f.status) f.status[0] = p.bad;
}

// BLK threads per workgroup.  ONE: a single workgroup takes all samples and
// finishes the sums itself (up to kNllOne samples: four per thread), instead of
// a second launch over the workgroups' partial sums.
template <int BLK, bool ONE>
__global__ __launch_bounds__(BLK) void k_nll_part(NllArgs a, NllFin f) {
    __shared__ double sl[BLK / kWave], sw[BLK / kWave];
    __shared__ int sb[BLK / kWave];
    double loss = 0.0, wsum = 0.0;
    int bad = 0;
    for (long long i = (long long)blockIdx.x * BLK + threadIdx.x; i < a.n; i += (long long)gridDim.x * BLK) {
        const long long t = a.t[i * a.ts];
        float li = 0.0f;
        if (t != a.ignore) {
            if (t < 0 || t >= a.c) {
                bad = 1;
            } else {
                const float w = a.w ? a.w[t] : 1.0f;
                li = -a.x[i * a.s0 + t * a.s1] * w;
                loss += (double)li;
                wsum += (double)w;
            }
        }
        if (a.reduction == 0) a.out[i] = li;
    }
    loss = wave_sum(loss);
    wsum = wave_sum(wsum);
    bad = wave_sum(bad);
    const int w = threadIdx.x / kWave;
    if (__lane_id() == 0) {
        sl[w] = loss;
        sw[w] = wsum;
        sb[w] = bad;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        NllPart p{0.0, 0.0, 0, 0};
        for (int k = 0; k < BLK / kWave; ++k) {
            p.loss += sl[k];
            p.weight += sw[k];
            p.bad |= sb[k] != 0;
        }
        if constexpr (ONE) nll_finish(f, p);
        else a.part[blockIdx.x] = p;
    }
}

__global__ __launch_bounds__(kNllBlock) void k_nll_fin(NllFin f) {
    __shared__ double sl[kNllBlock / kWave], sw[kNllBlock / kWave];
    __shared__ int sb[kNllBlock / kWave];
    double loss = 0.0, wsum = 0.0;
    int bad = 0;
    for (int k = threadIdx.x; k < f.nparts; k += kNllBlock) {
        loss += f.part[k].loss;
        wsum += f.part[k].weight;
        bad |= f.part[k].bad;
    }
    loss = wave_sum(loss);
    wsum = wave_sum(wsum);
    bad = wave_sum(bad);
    const int w = threadIdx.x / kWave;
    if (__lane_id() == 0) {
        sl[w] = loss;
        sw[w] = wsum;
        sb[w] = bad;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        NllPart p{0.0, 0.0, 0, 0};
        for (int k = 0; k < kNllBlock / kWave; ++k) {
            p.loss += sl[k];
            p.weight += sw[k];
            p.bad |= sb[k] != 0;
        }
        nll_finish(f, p);
    }
}

// ---- backward ---------------------------------------------------------------
struct NllBwdArgs {
    const float* g;
    long long gs;
    const long long* t;
    long long ts;
    const float* w;
    const float* tw;
    long long n, c, reduction, ignore;
    float* gi;
};

__device__ __forceinline__ float nll_grad_value(const NllBwdArgs& a, long long i, long long t) {
    float g = a.reduction == 0 ? a.g[i * a.gs] : a.g[0];
    if (a.reduction == 1 && a.tw) {
        const double tw = (double)a.tw[0];
        if (tw > 0.0) g = (float)((double)g / tw);
    }
    const float w = a.w ? a.w[t] : 1.0f;
    return -w * g;
}

// The dense [n, c] gradient is written as one flat run, one 16-byte store per
// thread (a write-only kernel runs fastest that way over a grid covering the
// output: measured on MI355X, a 256 MiB fill takes 40 us against 45-52 us with
// 2-8 stores per thread), so stores stay on 16 bytes whatever c is and a vector
// may hold the end of one row and the start of the next.  [4096, 50257]: one
// scalar store per thread took 377 us, vectors row by row (any alignment) 171,
// this 113 (7.3 TB/s); [4096, 32000] 78 -> 73.
__device__ __forceinline__ void nll_store(float* out, long long e, long long total, f32x4_t z) {
    if (e + 4 <= total) {
        __builtin_nontemporal_store(z, reinterpret_cast<f32x4_any*>(out + e));
    } else {
        for (int k = 0; e + k < total; ++k) out[e + k] = z[k];
    }
}

// Rows of at least 1024 elements: the 1024 elements of a workgroup lie in two
// rows at most.
__global__ __launch_bounds__(kNllBlock) void k_nll_bwd_rows(NllBwdArgs a) {
    const long long base = (long long)blockIdx.x * (4 * kNllBlock);
    const long long row = base / a.c;
    const long long col = base - row * a.c + 4 * threadIdx.x;  // may pass the row's end
    const long long total = a.n * a.c;
    if (base + 4 * threadIdx.x >= total) return;
    long long t0 = a.t[row * a.ts];
    if (t0 == a.ignore || t0 < 0 || t0 >= a.c) t0 = -4;
    long long t1 = row + 1 < a.n ? a.t[(row + 1) * a.ts] : a.ignore;
    t1 = (t1 == a.ignore || t1 < 0 || t1 >= a.c) ? -4 : t1 + a.c;
    f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
    if (t0 >= col && t0 < col + 4) {
        const float v = nll_grad_value(a, row, t0);
#pragma unroll
        for (int k = 0; k < 4; ++k) z[k] = t0 == col + k ? v : z[k];
    }
    if (t1 >= col && t1 < col + 4) {
        const float v = nll_grad_value(a, row + 1, t1 - a.c);
#pragma unroll
        for (int k = 0; k < 4; ++k) z[k] = t1 == col + k ? v : z[k];
    }
    nll_store(a.gi, base + 4 * threadIdx.x, total, z);
}

// Shorter rows (n * c < 2^32 - 1024): one 32-bit division per vector.  [8192,
// 1000]: one element per thread with a 64-bit division each took 12.7 us, this
// 6.7 us.
__global__ __launch_bounds__(kNllBlock) void k_nll_bwd_short(NllBwdArgs a) {
    const unsigned e = (blockIdx.x * (unsigned)kNllBlock + threadIdx.x) * 4u;
    const unsigned c = (unsigned)a.c, total = (unsigned)(a.n * a.c);
    if (e >= total) return;
    float z[4];
    nll_short_vector(e, c, total, a.ignore, [&](unsigned i) { return a.t[(long long)i * a.ts]; },
                     [&](unsigned i, long long t) { return nll_grad_value(a, i, t); }, z);
    nll_store(a.gi, e, total, f32x4_t{z[0], z[1], z[2], z[3]});
}

// Short rows beyond 32-bit indices: one element per thread over the
// flat [n, c] output.
__global__ __launch_bounds__(kNllBlock) void k_nll_bwd_flat(NllBwdArgs a) {
    const long long total = a.n * a.c;
    for (long long e = (long long)blockIdx.x * kNllBlock + threadIdx.x; e < total;
         e += (long long)gridDim.x * kNllBlock) {
        const long long row = e / a.c;
        const long long col = e - row * a.c;
        const long long t = a.t[row * a.ts];
        float v = 0.0f;
        if (t == col && t != a.ignore) v = nll_grad_value(a, row, t);
        a.gi[e] = v;
    }
}

}  // namespace
}  // namespace tpr

extern "C" size_t tpr_nll_loss_workspace_bytes(int64_t n) {
    using namespace tpr;
    if (n <= 0) return sizeof(NllPart);
    long long blocks = (n + kNllBlock - 1) / kNllBlock;
    if (blocks > kNllMaxBlocks) blocks = kNllMaxBlocks;
    return (size_t)blocks * sizeof(NllPart);
}

extern "C" int tpr_nll_loss(const void* input, int32_t dtype, int64_t n, int64_t c, int64_t s0, int64_t s1,
                            const int64_t* target, int64_t ts, const void* weight, int64_t reduction,
                            int64_t ignore_index, void* out, void* total_weight, int32_t* status,
                            void* workspace, size_t workspace_bytes, void* stream) {
    using namespace tpr;
    if (dtype != TPR_FLOAT32) return fail(TPR_ERR_UNSUPPORTED_DTYPE, "tpr_nll_loss: float32 input only");
    if (n < 0 || c < 0) return fail(TPR_ERR_INVALID_ARG, "tpr_nll_loss: negative extent");
    if (reduction < 0 || reduction > 2) return fail(TPR_ERR_INVALID_ARG, "tpr_nll_loss: invalid reduction mode");
    if (!total_weight || (!out && (reduction != 0 || n > 0)) || (n > 0 && (!input || !target)))
        return fail(TPR_ERR_INVALID_ARG, "tpr_nll_loss: null pointer");
    const size_t need = tpr_nll_loss_workspace_bytes(n);
    if (!workspace || workspace_bytes < need)
        return fail(TPR_ERR_WORKSPACE, "tpr_nll_loss: workspace smaller than tpr_nll_loss_workspace_bytes");
    hipStream_t st = static_cast<hipStream_t>(stream);
    NllPart* part = static_cast<NllPart*>(workspace);
    long long blocks = (n + kNllBlock - 1) / kNllBlock;
    if (blocks > kNllMaxBlocks) blocks = kNllMaxBlocks;
    if (blocks < 1) blocks = 1;
    NllArgs a{static_cast<const float*>(input), n, c, s0, s1,
              reinterpret_cast<const long long*>(target), ts, static_cast<const float*>(weight),
              reduction, ignore_index, static_cast<float*>(out), part};
    NllFin f{part, (int)blocks, reduction, static_cast<float*>(out), static_cast<float*>(total_weight),
             reinterpret_cast<int*>(status)};
    if (n <= kNllOne) {
        hipLaunchKernelGGL((k_nll_part<1024, true>), dim3(1), dim3(1024), 0, st, a, f);
        return check_launch("tpr_nll_loss");
    }
    hipLaunchKernelGGL((k_nll_part<kNllBlock, false>), dim3((unsigned)blocks), dim3(kNllBlock), 0, st, a, f);
    int rc = check_launch("tpr_nll_loss");
    if (rc) return rc;
    hipLaunchKernelGGL(k_nll_fin, dim3(1), dim3(kNllBlock), 0, st, f);
    return check_launch("tpr_nll_loss (finalize)");
}

extern "C" int tpr_nll_loss_backward(const void* grad_output, int64_t gs, const int64_t* target, int64_t ts,
                                     const void* weight, const void* total_weight, int64_t n, int64_t c,
                                     int64_t reduction, int64_t ignore_index, void* grad_input, void* stream) {
    using namespace tpr;
    if (n < 0 || c < 0) return fail(TPR_ERR_INVALID_ARG, "tpr_nll_loss_backward: negative extent");
    if (reduction < 0 || reduction > 2)
        return fail(TPR_ERR_INVALID_ARG, "tpr_nll_loss_backward: invalid reduction mode");
    if (n == 0 || c == 0) return TPR_OK;
    if (!grad_output || !target || !grad_input) return fail(TPR_ERR_INVALID_ARG, "tpr_nll_loss_backward: null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    NllBwdArgs a{static_cast<const float*>(grad_output), gs, reinterpret_cast<const long long*>(target), ts,
                 static_cast<const float*>(weight), static_cast<const float*>(total_weight),
                 n, c, reduction, ignore_index, static_cast<float*>(grad_input)};
    if (c >= 1024) {
        const long long blocks = (n * c + 4 * kNllBlock - 1) / (4 * kNllBlock);
        if (blocks > kMaxThreads / kNllBlock && n > 1) {  // 64 GiB of gradient: the samples in two halves
            const int64_t h = n / 2;
            const int rc = tpr_nll_loss_backward(grad_output, gs, target, ts, weight, total_weight, h, c, reduction,
                                                 ignore_index, grad_input, stream);
            if (rc != TPR_OK) return rc;
            return tpr_nll_loss_backward(a.g + (reduction == 0 ? h * gs : 0), gs, target + h * ts, ts, weight, total_weight,
                                         n - h, c, reduction, ignore_index, a.gi + h * c, stream);
        }
        if (blocks > kMaxThreads / kNllBlock) return fail(TPR_ERR_INVALID_ARG, "tpr_nll_loss_backward: too large");
        hipLaunchKernelGGL(k_nll_bwd_rows, dim3((unsigned)blocks), dim3(kNllBlock), 0, st, a);
    } else if (n * c < 0x100000000LL - 4 * kNllBlock) {
        const unsigned blocks = (unsigned)((n * c + 4 * kNllBlock - 1) / (4 * kNllBlock));
        hipLaunchKernelGGL(k_nll_bwd_short, dim3(blocks), dim3(kNllBlock), 0, st, a);
    } else {
        long long blocks = (n * c + kNllBlock - 1) / kNllBlock;
        const long long cap = (long long)device_info().cus * 32;
        if (blocks > cap) blocks = cap;
        hipLaunchKernelGGL(k_nll_bwd_flat, dim3((unsigned)blocks), dim3(kNllBlock), 0, st, a);
    }
    return check_launch("tpr_nll_loss_backward");
}
