// Host check of the estimated time of a permute against measured ones (MI355X, times of calls in
// a graph). Over the 260 that the rates were chosen from, estimate and time are within a factor
// of 1.7 of each other for tiles and a common fastest axis and of 3.5 for scattered sides; one rate
// for all of them would be off by up to 10.
#include <cstdio>
#include <vector>

#include "blas1.hpp"

using namespace ein;

struct Case {
    int bytes;
    std::vector<int64_t> dims; // row-major source
    std::vector<int32_t> perm; // axis i of the dense result is axis perm[i]
    double us;
    double factor;
};

int main() {
    std::vector<Case> const cases = {
        {8, {4, 160, 294, 16}, {0, 2, 3, 1}, 9.1, 1.7},
        {8, {3008, 236, 16}, {0, 2, 1}, 40.6, 1.7},
        {8, {150, 10, 62, 19}, {1, 3, 2, 0}, 10.6, 1.7},
        {4, {91, 507, 636}, {2, 1, 0}, 53.9, 1.7},
        {4, {56, 26, 5290}, {0, 2, 1}, 18.1, 1.7},
        {4, {83, 866, 23}, {2, 1, 0}, 8.5, 1.7},
        {8, {83, 283, 252}, {1, 0, 2}, 16.0, 1.7},
        {8, {7, 62, 51, 219}, {1, 2, 0, 3}, 16.0, 1.7},
        {8, {203, 45, 5, 27}, {0, 2, 1, 3}, 6.4, 1.7},
        {4, {24, 79, 2478}, {1, 0, 2}, 9.3, 1.7},
        {4, {395, 782, 19}, {1, 0, 2}, 17.5, 1.7},
        {4, {6, 9, 17, 44, 35}, {2, 0, 3, 1, 4}, 6.8, 1.7},
        {8, {23, 8, 6, 234, 6}, {0, 4, 3, 1, 2}, 11.1, 3.5},
        {8, {3, 181, 23, 217, 3}, {3, 2, 4, 0, 1}, 82.5, 3.5},
        {8, {59, 279, 10, 31}, {3, 1, 0, 2}, 97.7, 3.5},
        {4, {434, 3, 2617}, {0, 2, 1}, 11.2, 3.5},
        {4, {66, 8, 61, 44, 13}, {2, 1, 4, 3, 0}, 96.8, 3.5},
        {4, {53, 190, 61, 2, 11}, {4, 3, 0, 1, 2}, 175.2, 3.5},
    };
    int bad = 0;
    for (auto const &c : cases) {
        int const r = int(c.dims.size());
        std::vector<int64_t> sa(r, 1), sc(r, 1);
        for (int i = r - 1; i-- > 0;) {
            sa[i] = sa[i + 1] * c.dims[i + 1];
            sc[i] = sc[i + 1] * c.dims[c.perm[i + 1]];
        }
        double const us = permute_time_us(r, c.dims.data(), c.perm.data(), sa.data(), sc.data(), c.bytes);
        if (!(us < c.factor * c.us && us > c.us / c.factor)) {
            std::printf("%d bytes, first extent %lld: estimated %.1f us, measured %.1f\n", c.bytes, (long long)c.dims[0], us, c.us);
            ++bad;
        }
    }
    int64_t const none[2] = {0, 5}, one[2] = {1, 1}, s[2] = {5, 1};
    int32_t const id[2] = {0, 1};
    if (permute_time_us(2, none, id, s, s, 8) != 0.0 || !(permute_time_us(2, one, id, s, s, 8) > 0.0)) ++bad;
    if (!(permute_time_us(0, nullptr, nullptr, nullptr, nullptr, 8) > 0.0)) ++bad;
    std::printf("%d failures\n", bad);
    return bad != 0;
}
