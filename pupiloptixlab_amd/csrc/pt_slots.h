// Which frame and pixel a queue slot of a launch's camera paths holds, shared
// by the raygen kernel and the host tests (tests/slot_sim.cpp).
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define PT_SLOT_HD __host__ __device__ __forceinline__
#else
#define PT_SLOT_HD inline
#endif

namespace pupil {

// Frame (of the launch's `frames`) and place in the film's tile order of slot
// i: the launch's frames lie side by side, so a wave carries a few pixels in
// all of them.
PT_SLOT_HD void frame_slot(uint32_t frames, uint32_t i, uint32_t &frame, uint32_t &place) {
    frame = i % frames;
    place = i / frames;
}

// Pixel at place j of the tile order of a w x h film: full 8x8 tiles first,
// then the pixels of a partial right strip and bottom strip in row order.
PT_SLOT_HD uint32_t tiled_pixel(uint32_t j, uint32_t w, uint32_t h) {
    const uint32_t w8 = w & ~7u, h8 = h & ~7u, tiled = w8 * h8;
    if (j < tiled) {
        const uint32_t t = j >> 6, k = j & 63u, tiles_per_row = w8 >> 3;
        return ((t / tiles_per_row) * 8u + (k >> 3)) * w + (t % tiles_per_row) * 8u + (k & 7u);
    }
    j -= tiled;
    const uint32_t rw = w - w8;
    if (j < rw * h8) return (j / rw) * w + w8 + j % rw;
    return h8 * w + (j - rw * h8);
}

}  // namespace pupil
