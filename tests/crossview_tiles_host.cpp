// csrc/crossview_tiles.h on the host: the tiles hold every pixel, and none is empty; a
// strided loop passes the positions below its count, and ends.
#include <cstdint>
#include <cstdio>
#include <initializer_list>

#define __device__
#define __host__
#include "../multiviewdynrecon_amd/csrc/crossview_tiles.h"

using namespace mvdr;

int main() {
    const uint32_t counts[] = {1, 255, 2047, 2048, 2049, 921600, 4294836225u, 0xFFFFFFFFu - 2049, 0xFFFFFFFFu - 2047,
                               0xFFFFFFFFu - 300, 0xFFFFFFFFu - 255, 0xFFFFFFFEu};
    for (const uint32_t pixels : counts) {
        const uint64_t tiles = cv_tiles(pixels);
        const bool ok = tiles * kCvTile >= pixels && (tiles - 1) * kCvTile < pixels;
        if (!ok) {
            std::printf("%u pixels in %llu tiles\n", pixels, (unsigned long long)tiles);
            return 1;
        }
    }
    for (const uint32_t count : counts)
        for (const uint32_t step : {8192u, 131072u, 0x40000000u}) {
            // from the last positions, where the sum would pass 32 bits
            const uint32_t first = count > 4 * step && step < 0x40000000u ? count - 4 * step : 0;
            uint32_t i = first, steps = 1;
            while (steps < 8 && cv_step(i, step, count)) ++steps;
            const uint64_t want = (count - (uint64_t)first + step - 1) / step;
            if (steps != want || i != first + (want - 1) * step) {
                std::printf("count %u step %u: %u steps to %u\n", count, step, steps, i);
                return 1;
            }
        }
    return 0;
}
