// Traversal of the compressed wide BVH by persistent waves that keep their
// lanes busy: one ray per lane, and
//   - a lane whose ray has ended takes the next one of the wave's share as soon
//     as enough lanes are free, instead of waiting for the wave's slowest ray
//     (dynamic ray fetch, Aila and Laine, HPG 2009);
//   - leaf primitives are not tested where they are found.  The (lane,
//     primitive) pairs of the wave's rays gather in a ring in LDS and are
//     tested 64 at a time, one pair per lane, with the ray fetched from its
//     lane; a 64-bit minimum in LDS over (t, primitive id) -- the order that
//     defines the closest hit -- brings the results back together.
// The tree walk of a ray is trav_node / trav_next (pt_bvh.h) and so is the
// result: the pairs only change when a hit shortens its ray.
//
// Bound by VALU issue (97-100% busy alone).  With each wave walking 64 rays to
// the end and testing leaves in place, an instruction had 20 of 64 lanes at
// work on the terrain's rays and 30 in a closed room; now 43 and 45.  16
// bounces, shadow rays in launches of their own: terrain, 33 M paths, 28.7 ->
// 21.4 ms; closed room, 8.3 M paths, 19.7 -> 12.1 ms.  With them in the same
// launches 18.7 and 11.6 ms, 45 lanes in both.
#pragma once

#include <hip/hip_runtime.h>

#include "pt_bvh.h"

namespace pupil {

constexpr uint32_t kPairRing = 128;

// One wave's LDS.
template <int kEntries>
struct StreamLds {
    unsigned long long stack[kEntries][64];  // traversal stack, one column per lane
    unsigned long long key[64];              // best hit: t bits above, primitive id below
    float v[64], w[64], det[64];             // its undivided barycentrics
    uint2 pair[kPairRing];                   // leaf primitive, lane
};

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ uint32_t lane_rank(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
__device__ __forceinline__ float from_lane(float v, uint32_t src) {
    return u2f((uint32_t)__builtin_amdgcn_ds_bpermute((int)(4u * src), (int)f2u(v)));
}
__device__ __forceinline__ uint32_t from_lane(uint32_t v, uint32_t src) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(4u * src), (int)v);
}

// Free lanes that make the wave take new rays, and waiting rays (ended, pairs
// untested) that make it test what is there: a refill costs the wave a ray's
// set-up and its memory latency, a free lane its share of every instruction
// (8, 16 and 24: terrain 1080p, 64 frames, 86.5, 84.9 and 85.5 ms; closed room
// 640x360, 32 frames, 18.9, 18.3 and 18.6 ms).
constexpr uint32_t kRefillLanes = 16;
// Pairs that make the wave test them: a partly filled test wastes lanes, a
// late one lets its rays walk on past hits (24, 32, 40, 48 and 64: the same
// terrain 86.2, 85.3, 84.9, 85.0 and 85.3 ms; the room 18.6, 18.4, 18.3, 18.3 and
// 18.2 ms).  With no more rays to take, as many as rays in flight.
constexpr uint32_t kFlushPairs = 40;

// Traces `total` rays with all waves of the grid.  Wave `wave` starts with
// chunk `wave` of `chunk` rays and takes further chunks from the shared cursor
// (zero at launch).
// fetch(i, o, d, tmax, root, any_hit) reads ray i; t starts at `ext_tmin` for
// closest-hit and at `any_tmin` for any-hit rays, both positive.
// finish(i, any_hit, hit) takes its result (any-hit rays: only whether there
// is a hit).
template <bool kSph, int kEntries, typename Stack, typename LoadNode, typename Fetch, typename Finish>
__device__ __forceinline__ void trace_stream(StreamLds<kEntries> &L, Stack stack, const LeafTri *tris,
                                             LoadNode load_node, uint32_t total, uint32_t chunk,
                                             uint32_t wave, uint32_t waves, uint32_t *cursor, float ext_tmin,
                                             float any_tmin, Fetch fetch, Finish finish) {
    const uint32_t lane = __lane_id();
    uint32_t next = wave * chunk, end = min(next + chunk, total);
    if (next >= total) return;
    bool exhausted = false;
    uint32_t head = 0, count = 0;              // ring of pairs
    uint32_t appended = 0, tested = 0;         // pairs so far
    TravRay r;
    r.have = false;
    bool busy = false, any_hit = false;
    uint32_t ray = 0, last = 0;                // ray index; `appended` after its last pair
    uint32_t code = 0;                         // axes of the triangle test, bit 6: any hit

    auto test = [&](uint32_t n) {
        wave_sync();
        const uint2 pr = L.pair[(head + lane) & (kPairRing - 1u)];
        const bool on = lane < n;
        const uint32_t src = on ? pr.y : lane;
        const f3 o = mk3(from_lane(r.o.x, src), from_lane(r.o.y, src), from_lane(r.o.z, src));
        const uint32_t cd = from_lane(code, src);
        RayPre rp;
        rp.sx = from_lane(r.rp.sx, src);
        rp.sy = from_lane(r.rp.sy, src);
        rp.sz = from_lane(r.rp.sz, src);
        rp.kx = (int)(cd & 3u);
        rp.ky = (int)((cd >> 2) & 3u);
        rp.kz = (int)((cd >> 4) & 3u);
        f3 d = mk3(0.f);
        float tmax = 0.f;
        if (kSph) {
            d = mk3(from_lane(r.d.x, src), from_lane(r.d.y, src), from_lane(r.d.z, src));
            tmax = from_lane(r.tmax, src);
        }
        unsigned long long key = ~0ull;
        float V = 0.f, W = 0.f, det = 1.f;
        if (on) {
            const float4 *p = reinterpret_cast<const float4 *>(tris + pr.x);
            const float4 a = p[0], b = p[1], c = p[2];
            const float tmin = (cd & 64u) ? any_tmin : ext_tmin;
            float t;
            bool h;
            if (kSph && f2u(b.w) != 0u)
                h = intersect_sphere(o, d, f3{a.x, a.y, a.z}, b.x, tmin, tmax, t);
            else
                h = intersect_triangle(o, rp, f3{a.x, a.y, a.z}, f3{b.x, b.y, b.z}, f3{c.x, c.y, c.z}, t, V, W, det);
            // t >= tmin > 0: the order of float bits is that of the floats.
            if (h && t >= tmin) {
                const unsigned long long k = (unsigned long long)f2u(t) << 32 | f2u(a.w);
                if (k < L.key[src]) {
                    key = k;
                    atomicMin(&L.key[src], k);
                }
            }
        }
        wave_sync();
        if (key != ~0ull && L.key[src] == key) {
            L.v[src] = V;
            L.w[src] = W;
            L.det[src] = det;
        }
        wave_sync();
        head = (head + n) & (kPairRing - 1u);
        count -= n;
        tested += n;
        const unsigned long long best = L.key[lane];
        r.tbest = u2f((uint32_t)(best >> 32));
        if (any_hit && (uint32_t)best != 0xFFFFFFFFu) r.have = false;
    };

    for (;;) {
        // New rays for free lanes.
        const unsigned long long busy_m = __ballot(busy);
        const uint32_t in_flight = (uint32_t)__popcll(busy_m);
        if (!exhausted && (in_flight == 0u || in_flight + kRefillLanes <= 64u)) {
            if (next == end) {
                uint32_t c = 0;
                if (lane == 0) c = atomicAdd(cursor, 1u);
                c = (uint32_t)__builtin_amdgcn_readfirstlane((int)c) + waves;
                const unsigned long long begin = (unsigned long long)c * chunk;
                if (begin >= total) {
                    exhausted = true;
                } else {
                    next = (uint32_t)begin;
                    end = min(next + chunk, total);
                }
            }
            if (!exhausted) {
                const uint32_t n = min(64u - in_flight, end - next);
                const uint32_t rank = lane_rank(~busy_m);
                if (!busy && rank < n) {
                    ray = next + rank;
                    f3 o, d;
                    float tmax;
                    uint32_t root;
                    fetch(ray, o, d, tmax, root, any_hit);
                    const float tmin = any_hit ? any_tmin : ext_tmin;
                    Hit h;
                    stack.clear();
                    trav_init(r, load_node, o, d, tmin, tmax, stack, h, root);
                    code = (uint32_t)r.rp.kx | (uint32_t)r.rp.ky << 2 | (uint32_t)r.rp.kz << 4 | (any_hit ? 64u : 0u);
                    L.key[lane] = (unsigned long long)f2u(tmax) << 32 | 0xFFFFFFFFu;
                    if (!(tmax >= tmin)) {  // an empty range (a light closer than the shadow offset)
                        L.key[lane] = 0xFFFFFFFFull;
                        r.have = false;
                    }
                    busy = true;
                    last = tested;
                }
                next += n;
            }
        }
        if (__ballot(busy) == 0ull) {
            if (exhausted) break;
            continue;
        }
        // One node for each ray under way; its next node's load is in flight
        // while pairs are tested.
        uint32_t t_base = 0, t_bits = 0;
        if (r.have) {
            trav_node(r, t_base, t_bits);
            uint32_t node_index = 0;
            r.have = trav_next(r, stack, node_index);
            if (r.have) load_node(node_index, r.n);
        }
        for (unsigned long long m; (m = __ballot(t_bits != 0u)) != 0ull;) {
            const uint32_t n = (uint32_t)__popcll(m);
            if (t_bits) {
                const uint32_t k = (uint32_t)__builtin_ctz(t_bits);
                t_bits &= t_bits - 1u;
                L.pair[(head + count + lane_rank(m)) & (kPairRing - 1u)] = make_uint2(t_base + k, lane);
                last = appended + n;
            }
            count += n;
            appended += n;
            if (count >= 64u) test(64u);
        }
        const unsigned long long walking = __ballot(r.have);
        if (count && (count >= (exhausted ? min(in_flight + 1u, kFlushPairs) : kFlushPairs) || walking == 0ull ||
                      (uint32_t)__popcll(walking) + kRefillLanes <= (uint32_t)__popcll(__ballot(busy))))
            test(count);
        // Rays that have ended and whose pairs are all tested.
        if (busy && !r.have && (int32_t)(tested - last) >= 0) {
            const unsigned long long best = L.key[lane];
            Hit h;
            h.t = u2f((uint32_t)(best >> 32));
            h.prim = (uint32_t)best;
            h.b1 = h.b2 = 0.f;
            if (!any_hit && h.prim != 0xFFFFFFFFu) {
                h.b1 = L.v[lane] / L.det[lane];
                h.b2 = L.w[lane] / L.det[lane];
            }
            finish(ray, any_hit, h);
            busy = false;
        }
    }
}

}  // namespace pupil
