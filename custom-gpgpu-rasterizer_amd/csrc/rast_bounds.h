// rast_bounds.h -- the bounds that let a stage skip work: which boxes hold no
// triangle in view, which face test needs no square root, which pixels of a
// triangle's range cannot be covered.  Each claims something about values that
// the kernels evaluate in binary32, by margins of a few units in the last place;
// the functions compile for the host as well, where tests put them beside those
// evaluations.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace rast {

// The hardware reciprocal is within 1 ulp of 1 / x; the host takes the smaller
// neighbour of the rounded quotient, the harder case for edge_reach.
__host__ __device__ inline __attribute__((always_inline)) float approx_rcp(float x)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_rcpf(x);
#else
    return std::nextafter(1.f / x, 0.f);
#endif
}

__host__ __device__ inline __attribute__((always_inline)) void normalize3(float &x, float &y, float &z)
{
    const float m = sqrtf(x * x + y * y + z * z);
    if (m == 0.f) { x = 0.f; y = 0.f; z = 0.f; return; }
    const float inv = 1.f / m;
    x *= inv; y *= inv; z *= inv;
}

// Whether the face normal (fx, fy, fz), normalized as normalize3 does, makes a
// dot product above 0 (sign = 1) or below 0 (sign = -1) with the camera's
// forward c, decided as the binary32 evaluation decides it.  With s the dot
// product of the unnormalized normal, evaluated in binary32, T the sum of its
// terms' magnitudes and u = 2^-24: s is within 3.0001 u T of the exact product
// E, and the evaluated product of the normalized normal within 4.0001 u T inv
// of E inv (one rounding each in the scaled component and the term, two in the
// sum), so where |s| > 8 u T both have E's sign.  T > 1e-18 and components
// below 1e18 keep the squares and the products in range.  Elsewhere the
// normalized form itself is evaluated (a square root and a division).
__host__ __device__ inline __attribute__((always_inline)) bool faces(const float *c, float fx, float fy, float fz, float sign)
{
    const float p0 = c[0] * fx, p1 = c[1] * fy, p2 = c[2] * fz;
    const float s = (p0 + p1) + p2;
    const float T = (fabsf(p0) + fabsf(p1)) + fabsf(p2);
    if (fabsf(s) > T * (8.0f / 16777216.0f) && T > 1.0e-18f && fmaxf(fmaxf(fabsf(fx), fabsf(fy)), fabsf(fz)) < 1.0e18f)
        return s * sign > 0.f;
    normalize3(fx, fy, fz);
    const float cv = c[0] * fx + c[1] * fy + c[2] * fz;
    return sign > 0.f ? !(cv <= 0.f) : !(cv >= 0.f);
}

// How far left of (or above) a triangle's smallest corner coordinate a pixel
// of its range may lie and still pass the three evaluated edge tests.  A pixel
// d > 0 left of all corners has barycentric weights summing to 1 whose
// x-offsets, all at least d, sum to 0: the negative weights sum to at least
// d / w in magnitude (w, h the corners' extent), so one exact edge value is at
// most -A d / (2 w), A the exact |area|; with the opposite winding one is at
// most -A / 3.  The evaluated edge value is within 4.0002 u ((w + 2) h +
// (h + 2) w) <= 8.001 u (w + 2)(h + 2) of the exact one (u = 2^-24; the range
// reaches at most 2 pixels past the corners; roundings of the differences,
// the products and their difference), and area within 8.001 u w h of A.  So
// the pixel fails where d > 32.01 u max(w, 2)(w + 2)(h + 2) / area: an area
// too small to be trusted (below 16 u w h) makes that more than the 2 pixels
// in question, and as d <= 2 a larger one leaves A / 3 above the edge values'
// error.  34 u and the larger extent cover both axes and the roundings made
// here.
__host__ __device__ inline __attribute__((always_inline)) float edge_reach(float w, float h, float area)
{
    return (34.0f / 16777216.0f) * fmaxf(fmaxf(w, h), 2.f) * ((w + 2.f) * (h + 2.f)) * approx_rcp(area);
}

// The first pixel at or after lo that a triangle with smallest corner
// coordinate mn can cover: pixels before mn - reach - 2^-22 |mn| are passed
// over (the last term covers the rounding of the difference).
__host__ __device__ inline __attribute__((always_inline)) int first_pixel(float mn, float reach, int lo)
{
    return (int)ceilf(fmaxf(mn - (reach + fabsf(mn) * (4.0f / 16777216.0f)), (float)lo));
}

// A box [lo, hi] against the view volume of the clip matrix m (data[col][row]):
// every triangle with corners in it fails the evaluated frustum test if all its
// corners are outside one plane.  An evaluated clip coordinate is within 4.0003 u S
// of the exact affine value (S: its row's term magnitudes, largest over the box;
// u = 2^-24), its quotient by w within u more, and the values formed here, at
// the box's eight corners, within 4.0003 u S too: with all corners' w on one side
// of zero by 16 u Sw and, after multiplying by that sign, x + w, w - x and so on
// beyond 32 u (Sx + Sw), each evaluated quotient of every point of the box is on
// the far side of its plane.  A box reaching across w = 0, or with values that
// overflow or are not finite, is not culled.
//
// With twice these margins (scale 2) a box that is beyond a plane holds only
// boxes that are beyond it with them: the exact values at every point of it,
// within 4.0003 u S of the ones formed here, clear the single margins by more than
// the inner box's own error (the inner boxes' S are no larger).
struct BoxMargins {
    float x, y, z, w;
    bool fine;
};

__host__ __device__ inline __attribute__((always_inline)) BoxMargins box_margins(const float *m, float3 lo, float3 hi, float scale)
{
    const float u = 1.0f / 16777216.0f;
    const float ax = fmaxf(fabsf(lo.x), fabsf(hi.x)), ay = fmaxf(fabsf(lo.y), fabsf(hi.y));
    const float az = fmaxf(fabsf(lo.z), fabsf(hi.z));
    float S[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = fabsf(m[r]) * ax + fabsf(m[4 + r]) * ay + fabsf(m[8 + r]) * az + fabsf(m[12 + r]);
    BoxMargins g;
    g.fine = S[0] < 1.0e30f && S[1] < 1.0e30f && S[2] < 1.0e30f && S[3] < 1.0e30f;
    g.w = scale * (16.0f * u) * S[3] + scale * 1.0e-30f;
    g.x = scale * (32.0f * u) * (S[0] + S[3]);
    g.y = scale * (32.0f * u) * (S[1] + S[3]);
    g.z = scale * (32.0f * u) * (S[2] + S[3]);
    return g;
}

// The planes that the box's corner (x, y, z) is beyond; bits 6, 7: w > 0, w < 0.
__host__ __device__ inline __attribute__((always_inline)) uint32_t beyond_planes(const float *m, float x, float y, float z, const BoxMargins &g)
{
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = m[r] * x + m[4 + r] * y + m[8 + r] * z + m[12 + r];
    const float sg = v[3] < 0.f ? -1.f : 1.f, w = fabsf(v[3]);
    const float X = v[0] * sg, Y = v[1] * sg, Z = v[2] * sg;
    uint32_t b = 0;
    b |= X + w < -g.x ? 1u : 0u;
    b |= X - w > g.x ? 2u : 0u;
    b |= Y + w < -g.y ? 4u : 0u;
    b |= Y - w > g.y ? 8u : 0u;
    b |= Z < -g.z ? 16u : 0u;
    b |= Z - w > g.z ? 32u : 0u;
    b |= v[3] > g.w ? 64u : 0u;
    b |= v[3] < -g.w ? 128u : 0u;
    return b;
}

// Whether the box is out of view, from what all eight corners are beyond.
__host__ __device__ inline __attribute__((always_inline)) bool box_culled(uint32_t all, const BoxMargins &g) { return g.fine && (all & 0xC0u) != 0u && (all & 0x3Fu) != 0u; }

// The planes all eight corners are beyond, one after the other.
__host__ __device__ inline __attribute__((always_inline)) uint32_t box_beyond(const float *m, float3 lo, float3 hi, const BoxMargins &g)
{
    uint32_t all = 0xFFu;
#pragma unroll
    for (int c = 0; c < 8; ++c) all &= beyond_planes(m, c & 1 ? hi.x : lo.x, c & 2 ? hi.y : lo.y, c & 4 ? hi.z : lo.z, g);
    return all;
}

}  // namespace rast
