// CPU test of the nll_loss gradient's walk over short rows: every target and
// every weight that it reads lies in its array, and the values are those of
// the definition.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "nll_walk.h"

static long checks = 0;

static void run(unsigned n, unsigned c, long long last, long long ignore) {
    const unsigned total = n * c;
    std::vector<long long> t(n);
    for (unsigned i = 0; i < n; ++i) t[i] = (long long)((i * 5 + 2) % c);
    t[n / 2] = ignore;
    t[n - 1] = last;
    auto weight = [&](long long j) {
        if (j < 0 || j >= (long long)c) {
            std::printf("weight[%lld] read, n=%u c=%u last target %lld\n", j, n, c, last);
            std::exit(1);
        }
        return (float)(j + 1);
    };
    auto target = [&](unsigned i) {
        if (i >= n) {
            std::printf("target[%u] read, n=%u c=%u\n", i, n, c);
            std::exit(1);
        }
        return t[i];
    };
    auto value = [&](unsigned i, long long j) { return -weight(j) * (float)(i + 1); };
    for (unsigned e = 0; e < total; e += 4) {
        float z[4];
        tpr::nll_short_vector(e, c, total, ignore, target, value, z);
        for (unsigned k = 0; k < 4; ++k) {
            const unsigned row = (e + k) / c, col = (e + k) % c;
            const bool hit = e + k < total && t[row] == (long long)col && t[row] != ignore;
            const float want = hit ? -(float)(col + 1) * (float)(row + 1) : 0.0f;
            if (z[k] != want) {
                std::printf("element %u: %g, not %g (n=%u c=%u)\n", e + k, z[k], want, n, c);
                std::exit(1);
            }
            ++checks;
        }
    }
}

int main() {
    const long long ignored[] = {-100, 0, 3};
    for (unsigned c = 1; c <= 11; ++c)
        for (unsigned n = 1; n <= 9; ++n)
            for (long long ignore : ignored)
                for (long long last = -2; last <= (long long)c + 4; ++last) run(n, c, last, ignore);
    std::printf("OK %ld\n", checks);
    return 0;
}
