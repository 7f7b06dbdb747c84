"""The a-trous kernels at the edges of their tiles: spans of 64 pixels, groups
of four rows (images of half a million pixels and more) or one, strides wider
than the image, whole and real normal exponents, pixels without a surface and
pixels that are not finite; against the float64 restatement.
"""
import numpy as np
import pytest

import oracle.denoise as dn


def images(w, h, seed):
    rng = np.random.default_rng(seed)
    rgba = rng.gamma(2.0, 0.5, (h, w, 4)).astype(np.float32)
    alb = (0.2 + 0.05 * rng.random((h, w, 3))).astype(np.float32)
    n = np.array([0.1, 0.2, 1.0]) + 0.05 * rng.standard_normal((h, w, 3))
    n = (n / np.linalg.norm(n, axis=2, keepdims=True)).astype(np.float32)
    n[rng.random((h, w)) < 0.2] = 0.0
    return rgba, alb, n


# A weight's relative error is the normal product's rounding times the
# exponent, 64 x 2^-23 = 8e-6; the variance (a difference of moments, 25 x
# 2^-24 of the second) moves the luminance weight by less; five levels of
# normalized sums carry this on: 2e-4 bounds it with a factor of five.
@pytest.mark.gpu
@pytest.mark.parametrize("w,h,guides,exponent,levels", [
    (1, 1, "both", 64.0, 5), (3, 2, "both", 64.0, 10), (64, 4, "normal", 1.0, 5), (65, 9, "both", 48.0, 6),
    (63, 33, "both", 2.5, 5), (130, 71, "albedo", 64.0, 5), (1001, 501, "both", 64.0, 3), (1024, 489, "none", 64.0, 2),
    (999, 507, "normal", 3.0, 1), (40, 13001, "both", 7.3, 2)])
def test_tiles_and_exponents(tracer, w, h, guides, exponent, levels):
    print(f"case: denoise {w}x{h} guides={guides} exponent={exponent} levels={levels}", flush=True)
    rgba, a, n = images(w, h, w + h)
    a = a if guides in ("albedo", "both") else None
    n = n if guides in ("normal", "both") else None
    got = tracer.denoise_image(rgba, a, n, iterations=levels, sigma_normal=exponent)
    want = dn.denoise(rgba, a, n, iterations=levels, sigma_normal=exponent)
    assert np.allclose(got, want, rtol=2e-4, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(96, 40), (1000, 502)])
def test_pixels_that_are_not_finite_reach_their_windows_only(tracer, w, h):
    print(f"case: denoise {w}x{h} with an infinite and a NaN pixel", flush=True)
    rgba, a, n = images(w, h, 1)
    clean = tracer.denoise_image(rgba, a, n, iterations=1)
    rgba[9, 20, 0], rgba[30, 70, 1] = np.inf, np.nan
    got = tracer.denoise_image(rgba, a, n, iterations=1)
    assert not np.isfinite(got[9, 20, 0]) and not np.isfinite(got[30, 70, 1])
    near = np.zeros((h, w), bool)  # 2 pixels of taps see the variance of 1 more, taken from windows of 2 more
    near[4:15, 15:26] = near[25:36, 65:76] = True
    assert np.array_equal(got[~near], clean[~near])


# Sigmas whose square is below the float range (or zero in it): pixels of the
# same albedo blend, others do not, as in 64 bits.  No weight but the
# luminance's is rounded here, so the bound above holds.
@pytest.mark.gpu
@pytest.mark.parametrize("sigma", [1e-19, 1e-20, 3e-22, 1e-30])
@pytest.mark.parametrize("w,h", [(63, 33), (1000, 502)])
def test_albedo_scales_down_to_nothing(tracer, w, h, sigma):
    print(f"case: denoise {w}x{h} sigma_albedo={sigma}", flush=True)
    rgba, a, n = images(w, h, 7)
    a = np.where(a > 0.225, np.float32(0.25), np.float32(0.2))
    got = tracer.denoise_image(rgba, a, n, sigma_albedo=sigma)
    want = dn.denoise(rgba, a, n, sigma_albedo=sigma)
    assert np.allclose(got, want, rtol=2e-4, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("exponent", [64.0, 1.0, 0.01])
@pytest.mark.parametrize("w,h", [(63, 33), (1000, 502)])
def test_normals_without_length_are_no_surface(tracer, w, h, exponent):
    """A normal whose squared length underflows marks a pixel without a surface as a zero one does, bit for bit."""
    print(f"case: denoise {w}x{h} normals of 1e-24, exponent {exponent}", flush=True)
    rgba, a, n = images(w, h, 8)
    bare = ~n.any(-1)
    tiny = np.where(bare[..., None], np.float32(1e-24), n)
    assert np.array_equal(tracer.denoise_image(rgba, a, tiny, sigma_normal=exponent),
                          tracer.denoise_image(rgba, a, n, sigma_normal=exponent))
