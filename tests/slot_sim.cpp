// Host check of the queue order of camera paths
// (pupiloptixlab_amd/csrc/pt_slots.h), for the slot tests: over films of full
// and partial 8x8 tiles and launches of 1 to 64 frames, every (frame, pixel) is
// traced by exactly one slot.  Prints "ok" or the first failure.
#include <cstdio>
#include <vector>

#include "pt_slots.h"

using namespace pupil;

static bool check_launch(uint32_t frames, uint32_t w, uint32_t h) {
    const uint32_t npix = w * h, total = frames * npix;
    std::vector<uint8_t> seen(total, 0);
    for (uint32_t i = 0; i < total; ++i) {
        uint32_t f, place;
        frame_slot(frames, i, f, place);
        if (f >= frames || place >= npix) return false;
        const uint32_t pixel = tiled_pixel(place, w, h);
        if (pixel >= npix || seen[f * npix + pixel]) return false;
        seen[f * npix + pixel] = 1;
    }
    return true;  // as many slots as (frame, pixel) pairs, none twice
}

int main() {
    const uint32_t films[][2] = {{1, 1}, {7, 9}, {8, 8}, {9, 7}, {63, 1}, {1, 64}, {65, 33}, {97, 61}, {771, 433}, {1920, 1080}};
    const uint32_t frame_counts[] = {1u, 2u, 3u, 5u, 7u, 20u, 64u};
    for (const auto &film : films)
        for (uint32_t frames : frame_counts) {
            if ((uint64_t)frames * film[0] * film[1] > 50000000ull) continue;  // keep the host check fast
            if (!check_launch(frames, film[0], film[1])) {
                std::printf("slots failed: %u frames of %u x %u\n", frames, film[0], film[1]);
                return 1;
            }
        }
    std::printf("ok\n");
    return 0;
}
