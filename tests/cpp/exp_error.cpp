// The largest error of exp_table over [-32, 0], in units of the last place, against the 80-bit expl (tests/test_exp_table.py).
#include <cmath>
#include <cstdint>
#include <cstdio>

#include "../../ferro_amd/csrc/exp_table.hpp"

int main() {
    double2 pow2[64];
    for (int j = 0; j < 64; ++j) pow2[j] = {fs::exp_pow2[j][0], fs::exp_pow2[j][1]};
    long double worst = 0.0L;
    uint64_t x = 88172645463325252ull;
    for (int k = 0; k < 6000000; ++k) {
        x ^= x << 13; x ^= x >> 7; x ^= x << 17;
        const double f = (double)(x >> 11) * 0x1p-53;
        const double z = k % 3 == 0 ? -2.0 * f * f : k % 64 == 1 ? -(double)(x >> 59) : -32.0 * f;
        const long double want = expl((long double)z);
        int e;
        (void)std::frexp((double)want, &e);
        const long double err = fabsl(((long double)fs::exp_table(z, pow2) - want) / ldexpl(1.0L, e - 53));
        worst = err > worst ? err : worst;
    }
    std::printf("%.4Lf %d\n", worst, fs::exp_table(0.0, pow2) == 1.0 ? 1 : 0);
    return 0;
}
