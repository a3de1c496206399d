// The float32 quotient's short form (tode_math.h) on every pair of mantissas whose quotient lies within 2^-22 units of a
// rounding boundary: 2^k n = (2j + 1) d + s with |s| <= 8, for k = 24 (n >= d, quotient in [1, 2)) and k = 25 (n < d).
// For d = 2^a d' with d' odd, s = 2^a s' with s' odd and n is s' 2^(a - k) modulo d'.
// Prints: pairs looked at, pairs rounded to the wrong side.
#include <stdio.h>

#include "tode_math.h"

namespace host {
thread_local dim3 thread_idx, block_idx, grid_dim;
unsigned char *lds;
Barrier barrier;
}  // namespace host

int main() {
    const long long lo = 1 << 23, hi = 1 << 24;
    long long pairs = 0, wrong = 0;
    for (long long d = lo; d < hi; ++d) {
        const float r = 1.0f / (float)d;
        const int a = __builtin_ctzll(d);
        if (a > 3) continue;
        const long long odd = d >> a;
        for (int k = 24; k <= 25; ++k) {
            long long inverse = 1;  // 2^(a - k) modulo odd
            for (int i = 0; i < k - a; ++i) inverse = (inverse & 1 ? inverse + odd : inverse) / 2;
            for (long long s = -8 >> a; s <= 8 >> a; ++s) {
                if (!(s & 1)) continue;
                long long n = (s * inverse) % odd;
                if (n < 0) n += odd;
                const long long from = k == 24 ? d : lo, to = k == 24 ? hi : d;
                n += (from - n + odd - 1) / odd * odd;
                for (; n < to; n += odd) {
                    if (((((1ll << k) * n - s * (1ll << a)) / d) & 1) == 0) continue;  // (not next to a boundary but to a value)
                    ++pairs;
                    const float q = tode::quotient_with((float)n, (float)d, r);
                    wrong += q != (float)n / (float)d;
                }
            }
        }
    }
    printf("%lld %lld\n", pairs, wrong);
    return 0;
}
