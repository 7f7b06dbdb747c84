// Denoiser for the path tracer's output: the DenoisePass of the reference
// (system/denoise_pass.cpp:31-93) runs the closed OptiX AI denoiser
// (optix/denoiser.cpp) on the noisy buffer with optional albedo / normal
// guides and writes the "final result" buffer.  Here the filter is the
// edge-avoiding a-trous wavelet transform (Dammertz, Sewtz, Hanika, Lensch,
// HPG 2010) with the variance-guided luminance edge-stopping function of
// SVGF (Schied et al., HPG 2017), on albedo-demodulated color:
//
//   prepare   c = color / albedo (when albedo guides), l = luminance(c), and a
//             spatial luminance variance over a 5 x 5 window of pixels with a
//             similar normal / albedo;
//   k levels  5 x 5 B3-spline taps (1/16, 1/4, 3/8, 1/4, 1/16) at stride 2^k,
//             weight = h(x) h(y) w_l w_n w_a with
//               w_l = exp(-|l_p - l_q| / (sigma_l sqrt(g3x3(var_p)) + 1e-4)),
//               w_n = max(0, n_p . n_q)^sigma_n,
//               w_a = exp(-|a_p - a_q|^2 / sigma_a^2),
//             color' = sum w c / sum w, variance' = sum w^2 var / (sum w)^2;
//   finish    color x albedo.
//
// Each level is one stencil pass over HBM-resident float4 images, the last one
// multiplying the albedo back.  A level is bound by its arithmetic (25 taps a
// pixel, each with a normal and an albedo weight) and then by the taps' loads
// through L1, so:
//   - a lane filters kRows pixels that lie `step` rows apart: each loaded tap
//     serves up to kRows of them, 10 taps a pixel instead of 25 at four;
//   - a wave covers 64 neighbouring pixels of a row, so every load is
//     contiguous and the row tests are scalar;
//   - the weights share one exponential, and whole normal exponents are
//     products.
// 1080p, all guides: 244 us a level with a lane per pixel and powf, 107 so;
// the call with its read-back 3390 -> 2570 us.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>

#include "pt_denoise.h"
#include "pt_math.h"

namespace pupil {
namespace {

constexpr uint32_t kLanes = 64, kWaves = 4;  // a block filters kWaves groups of rows, 64 pixels wide

struct Guides {
    const float *albedo;  // 3 floats per pixel, or null
    const float *normal;  // 3 floats per pixel, or null
};

// How the normal weight's exponent is applied.
enum NormalPower { kNoNormal = 0, kWholePower, kRealPower };
constexpr float kMaxWholePower = 1024.f;

// Images below this many pixels give a lane one row: four would leave fewer
// than two waves for each of the 1024 SIMDs.
constexpr uint64_t kFewPixels = 500000;

__device__ __forceinline__ f3 load3(const float *p, size_t i) { return mk3(p[3 * i], p[3 * i + 1], p[3 * i + 2]); }
__device__ __forceinline__ float dot_fma(f3 a, f3 b) { return fmaf(a.x, b.x, fmaf(a.y, b.y, a.z * b.z)); }
__device__ __forceinline__ float luminance_fma(f3 c) { return dot_fma(c, mk3(0.2126f, 0.7152f, 0.0722f)); }
__device__ __forceinline__ f3 demodulate(f3 c, f3 a) {
    return mk3(c.x / fmaxf(a.x, kDenoiseAlbedoEps), c.y / fmaxf(a.y, kDenoiseAlbedoEps),
               c.z / fmaxf(a.z, kDenoiseAlbedoEps));
}

// 1 / sigma^2 of the albedo weight.  Finite, so that equal albedos weigh 1: the
// reciprocal overflows for sigma below 5.4e-20, where only differences under
// 1e-18 weigh anything else than 0.
__device__ __forceinline__ float inverse_square(float sigma) { return fminf(1.f / (sigma * sigma), FLT_MAX); }

// e^-x as one exp2 (argument and result each rounded once).
__device__ __forceinline__ float exp_neg(float x) { return __builtin_amdgcn_exp2f(x * -1.44269504088896341f); }

// max(0, n . nq[k])^exponent by the exponent's class.  A whole exponent takes
// one product per doubling (the default, 64, six; powf costs about eighty
// instructions).  The exponent scales the cosine's rounding, so both are taken
// in double and the weight rounds once, in no more time (1080p, a level: 105
// us in float, 107 in double; a noisy image against 64 bits: 2.5e-7 with a
// float cosine and powf, 1.4e-7 so).
template <int kNormal, int kRows, typename Guide>
__device__ __forceinline__ void normal_weights(const Guide (&gp)[kRows], f3 nq, int lo, int hi, float exponent,
                                               float (&wn)[kRows]) {
    if constexpr (kNormal == kWholePower) {
        const double qx = nq.x, qy = nq.y, qz = nq.z;
        double d[kRows];
#pragma unroll
        for (int k = 0; k < kRows; ++k)
            if (k >= lo && k <= hi)
                d[k] = fmax(0.0, fma((double)gp[k].n.x, qx, fma((double)gp[k].n.y, qy, (double)gp[k].n.z * qz)));
        uint32_t e = (uint32_t)exponent;
        while ((e & 1u) == 0u) {
#pragma unroll
            for (int k = 0; k < kRows; ++k)
                if (k >= lo && k <= hi) d[k] *= d[k];
            e >>= 1;
        }
#pragma unroll
        for (int k = 0; k < kRows; ++k)
            if (k >= lo && k <= hi) {
                double r = d[k];
                for (uint32_t rest = e >> 1; rest; rest >>= 1) {
                    d[k] *= d[k];
                    if (rest & 1u) r *= d[k];
                }
                wn[k] = (float)r;
            }
    } else if constexpr (kNormal == kRealPower) {
#pragma unroll
        for (int k = 0; k < kRows; ++k)
            if (k >= lo && k <= hi) wn[k] = powf(fmaxf(0.f, dot_fma(gp[k].n, nq)), exponent);
    }
}

// What the weights need of a pixel.
struct GuideValue {
    f3 n, a;
    bool bare;  // no surface: a zero normal
};

template <int kNormal, bool kAlbedo>
__device__ __forceinline__ GuideValue load_guides(const Guides &g, size_t p) {
    GuideValue v;
    v.bare = false;
    if constexpr (kNormal != kNoNormal) {
        v.n = load3(g.normal, p);
        v.bare = dot(v.n, v.n) == 0.f;
        if (v.bare) v.n = mk3(0.f);  // also where only the square is zero: no weight against a surface
    }
    if constexpr (kAlbedo) v.a = load3(g.albedo, p);
    return v;
}

// A tap: its pixel and what the weights need of it.
struct Tap {
    float4 c;
    GuideValue g;
};

// The 5 x 5 windows at stride `step` of a lane's rows y0, y0 + step, ...:
// calls use(i, row, tap) for each tap column i and window row in bounds, which
// serves the rows k with 0 <= row - k <= 4.  A row's loads are issued before
// the row above it is used.
template <int kNormal, bool kAlbedo, int kRows, typename Use>
__device__ __forceinline__ void for_taps(const float4 *in, const Guides &g, int x, int y0, int w, int h, int step,
                                         const Use &use) {
    for (int i = 0; i < 5; ++i) {
        const int qx = x + (i - 2) * step;
        if (qx < 0 || qx >= w) continue;
        const auto load = [&](int row) {
            const size_t q = (size_t)min(max(y0 + (row - 2) * step, 0), h - 1) * w + qx;
            return Tap{in[q], load_guides<kNormal, kAlbedo>(g, q)};
        };
        Tap next = load(0);
#pragma unroll
        for (int row = 0; row < kRows + 4; ++row) {
            const Tap t = next;
            if (row < kRows + 3) next = load(row + 1);
            const int qy = y0 + (row - 2) * step;
            if (qy >= 0 && qy < h) use(i, row, t);
        }
    }
}

// The 64-pixel span and the first row of this wave: tiles in row-major order,
// each XCD (blocks go round them) a contiguous part, so that neighbouring
// rows' taps meet in one L2.  A group's rows lie `step` apart.
template <int kRows>
__device__ __forceinline__ bool wave_place(uint32_t w, uint32_t h, uint32_t log2_step, uint32_t blocks, int &x0, int &y0) {
    const uint32_t per = (blocks + 7u) / 8u, tile = (blockIdx.x % 8u) * per + blockIdx.x / 8u;
    const uint32_t wide = (w + kLanes - 1u) / kLanes;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / kLanes));
    const uint32_t r = tile / wide * kWaves + wave;
    x0 = (int)(tile % wide * kLanes);
    const uint64_t y = (((uint64_t)(r >> log2_step) * kRows) << log2_step) + (r & ((1u << log2_step) - 1u));
    y0 = (int)y;
    return tile < blocks && y < h;
}

// Demodulated color (xyz) and the spatial luminance variance (w).
template <int kNormal, bool kAlbedo, int kRows>
__global__ __launch_bounds__(256) void k_dn_prepare(const float4 *in, Guides g, float4 *out, uint32_t w, uint32_t h,
                                                    uint32_t blocks, DenoiseParams prm) {
    int x0, y0;
    if (!wave_place<kRows>(w, h, 0u, blocks, x0, y0)) return;
    const int x = min(x0 + (int)__lane_id(), (int)w - 1);
    const float inv_albedo = inverse_square(prm.sigma_albedo);
    GuideValue gp[kRows];
    // Moments about the center's luminance: their difference loses nothing
    // where the window is flat.
    f3 cp[kRows];
    float lp[kRows], s1[kRows], s2[kRows], sw[kRows];
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        const size_t p = (size_t)min(y0 + k, (int)h - 1) * w + x;
        gp[k] = load_guides<kNormal, kAlbedo>(g, p);
        const float4 c4 = in[p];
        cp[k] = mk3(c4.x, c4.y, c4.z);
        if constexpr (kAlbedo) cp[k] = demodulate(cp[k], gp[k].a);
        lp[k] = luminance_fma(cp[k]);
        s1[k] = s2[k] = sw[k] = 0.f;
    }
    for_taps<kNormal, kAlbedo, kRows>(in, g, x, y0, (int)w, (int)h, 1, [&](int, int row, const Tap &t) {
        const float4 c4 = t.c;
        const GuideValue &gq = t.g;
        f3 c = mk3(c4.x, c4.y, c4.z);
        if constexpr (kAlbedo) c = demodulate(c, gq.a);
        const float l = luminance_fma(c);
        const int lo = max(row - 4, 0), hi = min(row, kRows - 1);
        float wn[kRows];
        normal_weights<kNormal>(gp, gq.n, lo, hi, prm.sigma_normal, wn);
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            if (k < lo || k > hi) continue;
            float wq = 1.f;
            // Pixels without a surface only blend with each other.
            if constexpr (kNormal != kNoNormal) wq = gp[k].bare && gq.bare ? 1.f : wn[k];
            if constexpr (kAlbedo) {
                const f3 da = gp[k].a - gq.a;
                const float e = dot_fma(da, da) * inv_albedo;
                wq *= exp_neg(gp[k].bare != gq.bare ? 0.f : e);
            }
            const float dl = l - lp[k], wl = wq * dl;
            s1[k] += wl;
            s2[k] = fmaf(wl, dl, s2[k]);
            sw[k] += wq;
        }
    });
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        if (y0 + k >= (int)h || x0 + (int)__lane_id() >= (int)w) break;
        const float m1 = s1[k] / sw[k], m2 = s2[k] / sw[k];
        out[(size_t)(y0 + k) * w + x] = make_float4(cp[k].x, cp[k].y, cp[k].z, fmaxf(0.f, fmaf(-m1, m1, m2)));
    }
}

// One a-trous level at stride 2^log2_step; the last one remodulates.
template <int kNormal, bool kAlbedo, int kRows>
__global__ __launch_bounds__(256) void k_dn_atrous(const float4 *in, Guides g, float4 *out, uint32_t w, uint32_t h,
                                                   uint32_t log2_step, uint32_t last, uint32_t blocks,
                                                   DenoiseParams prm) {
    int x0, y0;
    if (!wave_place<kRows>(w, h, log2_step, blocks, x0, y0)) return;
    const int step = 1 << log2_step, lane = (int)__lane_id();
    const int x = min(x0 + lane, (int)w - 1);
    const float inv_albedo = inverse_square(prm.sigma_albedo);
    GuideValue gp[kRows];
    float l0[kRows], inv_sigma[kRows], sv[kRows], sw[kRows];
    f3 sc[kRows];
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        const int y = min(y0 + k * step, (int)h - 1);
        const size_t p = (size_t)y * w + x;
        gp[k] = load_guides<kNormal, kAlbedo>(g, p);
        const float4 c = in[p];
        l0[k] = luminance_fma(mk3(c.x, c.y, c.z));
        // 3 x 3 Gaussian (1/4, 1/2, 1/4) of the variance at the center.
        float gv = 0.f, gw = 0.f;
#pragma unroll
        for (int dy = -1; dy <= 1; ++dy) {
            if (y + dy < 0 || y + dy >= (int)h) continue;
            const float4 *r = in + (size_t)(y + dy) * w;
            const float ky = dy == 0 ? 0.5f : 0.25f;
#pragma unroll
            for (int dx = -1; dx <= 1; ++dx) {
                if (x + dx < 0 || x + dx >= (int)w) continue;
                const float kxy = ky * (dx == 0 ? 0.5f : 0.25f);
                gv = fmaf(kxy, r[x + dx].w, gv);
                gw += kxy;
            }
        }
        inv_sigma[k] = 1.f / (prm.sigma_luminance * sqrtf(gv / gw) + 1e-4f);
        sc[k] = mk3(0.f);
        sv[k] = sw[k] = 0.f;
    }
    for_taps<kNormal, kAlbedo, kRows>(in, g, x, y0, (int)w, (int)h, step, [&](int i, int row, const Tap &t) {
        const float4 cq = t.c;
        const GuideValue &gq = t.g;
        const float lq = luminance_fma(mk3(cq.x, cq.y, cq.z));
        const float ki = i == 2 ? 3.f / 8.f : (i == 1 || i == 3 ? 1.f / 4.f : 1.f / 16.f);
        const int lo = max(row - 4, 0), hi = min(row, kRows - 1);
        float wn[kRows];
        normal_weights<kNormal>(gp, gq.n, lo, hi, prm.sigma_normal, wn);
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            if (k < lo || k > hi) continue;
            const int j = row - k;
            const float kj = j == 2 ? 3.f / 8.f : (j == 1 || j == 3 ? 1.f / 4.f : 1.f / 16.f);
            float e = fabsf(l0[k] - lq) * inv_sigma[k];
            if constexpr (kAlbedo) {
                const f3 da = gp[k].a - gq.a;
                e += gp[k].bare != gq.bare ? 0.f : dot_fma(da, da) * inv_albedo;
            }
            float wq = ki * kj * exp_neg(e);
            if constexpr (kNormal != kNoNormal) wq *= gp[k].bare && gq.bare ? 1.f : wn[k];
            sc[k] = mk3(fmaf(wq, cq.x, sc[k].x), fmaf(wq, cq.y, sc[k].y), fmaf(wq, cq.z, sc[k].z));
            sv[k] = fmaf(wq * wq, cq.w, sv[k]);
            sw[k] += wq;
        }
    });
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        const int y = y0 + k * step;
        if (y >= (int)h || x0 + lane >= (int)w) break;
        f3 r = mk3(sc[k].x / sw[k], sc[k].y / sw[k], sc[k].z / sw[k]);
        float v = sv[k] / (sw[k] * sw[k]);
        if (last) {
            if constexpr (kAlbedo)
                r = mk3(r.x * fmaxf(gp[k].a.x, kDenoiseAlbedoEps), r.y * fmaxf(gp[k].a.y, kDenoiseAlbedoEps),
                        r.z * fmaxf(gp[k].a.z, kDenoiseAlbedoEps));
            v = 1.f;
        }
        out[(size_t)y * w + x] = make_float4(r.x, r.y, r.z, v);
    }
}

// Blocks that cover the groups of kRows rows at stride 2^log2_step.
uint32_t dn_blocks(uint32_t w, uint32_t h, uint32_t rows, uint32_t log2_step) {
    const uint64_t band = (uint64_t)rows << log2_step;
    const uint64_t groups = ((h + band - 1) / band) << log2_step;
    return (uint32_t)((w + kLanes - 1) / kLanes * ((groups + kWaves - 1) / kWaves));
}

template <int kNormal, bool kAlbedo, int kRows>
void dn_enqueue(hipStream_t stream, uint32_t w, uint32_t h, const float4 *in, const Guides &g, float4 *out, float4 *a,
                float4 *b, const DenoiseParams &prm) {
    const dim3 block(kLanes * kWaves);
    uint32_t blocks = dn_blocks(w, h, kRows, 0u);
    hipLaunchKernelGGL((k_dn_prepare<kNormal, kAlbedo, kRows>), dim3((blocks + 7u) / 8u * 8u), block, 0, stream, in, g,
                       a, w, h, blocks, prm);
    for (uint32_t k = 0; k < prm.iterations; ++k) {
        const uint32_t last = k + 1 == prm.iterations;
        blocks = dn_blocks(w, h, kRows, k);
        hipLaunchKernelGGL((k_dn_atrous<kNormal, kAlbedo, kRows>), dim3((blocks + 7u) / 8u * 8u), block, 0, stream, a,
                           g, last ? out : b, w, h, k, last, blocks, prm);
        float4 *t = a;
        a = b;
        b = t;
    }
}

template <int kRows>
void dn_select(hipStream_t stream, uint32_t w, uint32_t h, const float4 *in, const Guides &g, float4 *out, float4 *a,
               float4 *b, const DenoiseParams &prm) {
    const float e = prm.sigma_normal;
    const int normal = !g.normal ? kNoNormal : (e >= 1.f && e <= kMaxWholePower && e == floorf(e) ? kWholePower : kRealPower);
    const auto run = [&](auto fn) { fn(stream, w, h, in, g, out, a, b, prm); };
    if (g.albedo) {
        if (normal == kNoNormal) run(dn_enqueue<kNoNormal, true, kRows>);
        else if (normal == kWholePower) run(dn_enqueue<kWholePower, true, kRows>);
        else run(dn_enqueue<kRealPower, true, kRows>);
    } else {
        if (normal == kNoNormal) run(dn_enqueue<kNoNormal, false, kRows>);
        else if (normal == kWholePower) run(dn_enqueue<kWholePower, false, kRows>);
        else run(dn_enqueue<kRealPower, false, kRows>);
    }
}

}  // namespace

hipError_t denoise_launch(hipStream_t stream, uint32_t w, uint32_t h, const float4 *in, const float *albedo,
                          const float *normal, float4 *out, float4 *scratch, const DenoiseParams &prm) {
    const Guides g{albedo, normal};
    float4 *a = scratch, *b = scratch + (size_t)w * h;
    if ((uint64_t)w * h >= kFewPixels) dn_select<4>(stream, w, h, in, g, out, a, b, prm);
    else dn_select<1>(stream, w, h, in, g, out, a, b, prm);
    return hipGetLastError();
}

}  // namespace pupil
