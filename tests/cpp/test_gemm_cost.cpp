// Host check of the estimated time of a dense product, which decides between packing a
// generic contraction's operands and gathering them: it holds for both types, for every tile
// that a call may take, and is never below what the product's flops take at the peak rate.
#include <cmath>
#include <cstdio>
#include <random>

#include "gemm.hpp"

using namespace ein;

int main() {
    int bad = 0;
    std::mt19937_64 rng(7);
    auto draw = [&](double lo, double hi) {
        return int64_t(std::exp(std::uniform_real_distribution<>(std::log(lo), std::log(hi))(rng)));
    };
    double const peak[] = {78.6e6, 157.3e6}; // flops per us
    for (int it = 0; it < 20000; ++it) {
        int64_t const m = draw(1, 6000), n = draw(1, 6000), k = draw(1, 20000), batch = it % 3 ? 1 : draw(1, 100);
        for (int eb : {8, 4})
            for (bool krow : {false, true})
                for (int unaligned : {0, 1, 2}) {
                    double const us    = gemm_time_us(m, n, k, batch, eb, krow, unaligned);
                    double const least = 2.0 * double(m) * double(n) * double(k) * double(batch) / peak[eb == 4];
                    if (!(us > 1.0 && us >= least && std::isfinite(us)) && bad++ < 8)
                        std::printf("%lld x %lld x %lld, batch %lld, %d bytes, krow %d, unaligned %d: %g us, at least %g\n",
                                    (long long)m, (long long)n, (long long)k, (long long)batch, eb, int(krow), unaligned, us, least);
                }
    }
    std::printf("%d failures\n", bad);
    return bad != 0;
}
