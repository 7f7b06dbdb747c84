// Exchange within groups of eight neighbouring lanes (all eight active): with
// lane ^ 1 and lane ^ 2 of the quad, then with the mirrored lane of the other
// quad.
#pragma once

#include <hip/hip_runtime.h>

#include "pt_math.h"

namespace pupil {

template <typename Op>
__device__ __forceinline__ uint32_t group_reduce(uint32_t v, Op op) {
    v = op(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true));
    v = op(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true));
    return op(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, true));
}
__device__ __forceinline__ float group_min(float v) {
    return u2f(group_reduce(f2u(v), [](uint32_t a, uint32_t b) { return f2u(fminf(u2f(a), u2f(b))); }));
}
__device__ __forceinline__ float group_max(float v) {
    return u2f(group_reduce(f2u(v), [](uint32_t a, uint32_t b) { return f2u(fmaxf(u2f(a), u2f(b))); }));
}
__device__ __forceinline__ bool group_all(bool p) {
    return group_reduce(p ? 1u : 0u, [](uint32_t a, uint32_t b) { return a & b; }) != 0u;
}

}  // namespace pupil
