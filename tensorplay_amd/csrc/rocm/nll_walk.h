// The walk of one vector of the nll_loss gradient over short rows, apart from
// the kernel so that its reads can be checked on the CPU.
#pragma once

#ifdef __HIPCC__
#define TPR_WALK __device__ __forceinline__
#else
#define TPR_WALK inline
#endif

namespace tpr {

// z[0..3] for the elements e .. e + 3 of the flat [n, c] gradient (e < total =
// n * c): target(i) is sample i's target (below 0 or at least c: ignored, or
// out of range and without a column), value(i, t) the gradient at its column t.
// Elements at total and beyond have no row: they keep their 0.
template <class Target, class Value>
TPR_WALK void nll_short_vector(unsigned e, unsigned c, unsigned total, long long ignore, Target&& target,
                               Value&& value, float (&z)[4]) {
    unsigned row = e / c, col = e - row * c;
    long long t = target(row);
#pragma GCC unroll 4
    for (int k = 0; k < 4; ++k) {
        z[k] = 0.0f;
        if (t == (long long)col && t != ignore) z[k] = value(row, t);
        if (++col == c) {
            // past the last row's end no column follows, whatever its target is
            const bool more = e + k + 1 < total;
            if (more) col = 0;
            t = more ? target(++row) : -1;
        }
    }
}

}  // namespace tpr
