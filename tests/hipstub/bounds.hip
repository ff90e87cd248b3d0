// The kernels' bounds (rast_bounds.h) as host functions over arrays.
#include "rast_bounds.h"

using namespace rast;

// The planes a box is beyond at margins scaled by `scale`, 0 where it is not culled.
extern "C" void bounds_box(size_t n, const float *m, const float *lo, const float *hi, float scale, uint32_t *planes)
{
    for (size_t i = 0; i < n; ++i, m += 16, lo += 3, hi += 3) {
        const float3 a = make_float3(lo[0], lo[1], lo[2]), c = make_float3(hi[0], hi[1], hi[2]);
        const BoxMargins g = box_margins(m, a, c, scale);
        const uint32_t all = box_beyond(m, a, c, g);
        planes[i] = box_culled(all, g) ? all & 0x3Fu : 0u;
    }
}

extern "C" void bounds_reach(size_t n, const float *w, const float *h, const float *area, float *reach)
{
    for (size_t i = 0; i < n; ++i) reach[i] = edge_reach(w[i], h[i], area[i]);
}

extern "C" void bounds_first(size_t n, const float *mn, const float *reach, const int *lo, int *first)
{
    for (size_t i = 0; i < n; ++i) first[i] = first_pixel(mn[i], reach[i], lo[i]);
}

extern "C" void bounds_faces(size_t n, const float *c, const float *f, float sign, uint8_t *yes)
{
    for (size_t i = 0; i < n; ++i, c += 3, f += 3) yes[i] = faces(c, f[0], f[1], f[2], sign);
}
