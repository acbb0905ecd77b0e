// csrc/crossview_tiles.h on the host: the tiles hold every pixel, and none is empty.
#include <cstdint>
#include <cstdio>

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
    return 0;
}
