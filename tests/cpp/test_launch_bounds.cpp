// Host check that long tile lists of the wave kernels go in launches that HIP takes whole:
// consecutive parts, all tiles in them once, each of fewer than 2^32 threads.
#include <cstdio>

#include "wave_tile.hpp"

using namespace ein;

int main() {
    int bad = 0;
    for (uint64_t ntiles : {uint64_t{0}, uint64_t{1}, uint64_t{WAVE_TILES_MAX} - 1, uint64_t{WAVE_TILES_MAX}, uint64_t{WAVE_TILES_MAX} + 1,
                            uint64_t{1} << 26, uint64_t{0x7fffffff}, uint64_t{0xffffffff}}) {
        uint64_t next = 0;
        int const st  = for_wave_parts(uint32_t(ntiles), [&](uint32_t first, uint32_t count) {
            if (first != next || count == 0 || (uint64_t(count) + 3) / 4 * GEMM_THREADS >= (uint64_t{1} << 32)) ++bad;
            next = uint64_t(first) + count;
            return next > ntiles ? 1 : 0;
        });
        if (st != 0 || next != ntiles) {
            std::printf("%llu of %llu tiles launched\n", (unsigned long long)next, (unsigned long long)ntiles);
            ++bad;
        }
    }
    // a failed part ends the list
    int calls = 0;
    if (for_wave_parts(0xffffffffu, [&](uint32_t, uint32_t) { return ++calls == 2 ? 7 : 0; }) != 7 || calls != 2) ++bad;
    std::printf("%d failures\n", bad);
    return bad != 0;
}
