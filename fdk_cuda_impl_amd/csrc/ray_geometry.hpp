// Device-side ray setup shared by the projection kernels and their transposes.
#pragma once

#include <hip/hip_runtime.h>

#include "yk_internal.hpp"

namespace yk {
namespace {

struct AxisInfo {
    int p0, p1, p2;     // component index of c0, c1, c2
    int n0, n1, n2;
    float v0, v1, v2;
};

__device__ __forceinline__ AxisInfo axis_info(int axis, const VolumeGeom& g)
{
    AxisInfo a;
    if (axis == 0) { a.p0 = 0; a.p1 = 1; a.p2 = 2; a.n0 = g.nx; a.n1 = g.ny; a.n2 = g.nz; a.v0 = g.vx; a.v1 = g.vy; a.v2 = g.vz; }
    else if (axis == 1) { a.p0 = 1; a.p1 = 0; a.p2 = 2; a.n0 = g.ny; a.n1 = g.nx; a.n2 = g.nz; a.v0 = g.vy; a.v1 = g.vx; a.v2 = g.vz; }
    else { a.p0 = 2; a.p1 = 0; a.p2 = 1; a.n0 = g.nz; a.n1 = g.nx; a.n2 = g.ny; a.v0 = g.vz; a.v1 = g.vx; a.v2 = g.vy; }
    return a;
}

template <typename T>
__device__ __forceinline__ T pick(int k, T a, T b, T c) { return k == 0 ? a : (k == 1 ? b : c); }

struct JRay {
    float a1, b1, a2, b2, L;
};

// Per-ray Joseph line in volume-centred voxel units.  Shared by the forward
// kernel and the transpose's ray table, with contraction disabled so both
// evaluate the same IEEE operations and obtain bit-identical parameters.
__device__ __forceinline__ bool joseph_ray(const ProjViewDev& pv, const AxisInfo& ax,
    int u, int v, JRay& r)
{
#pragma clang fp contract(off)
    const float dx = (pv.detS[0] + float(u) * pv.detU[0]) + float(v) * pv.detV[0];
    const float dy = (pv.detS[1] + float(u) * pv.detU[1]) + float(v) * pv.detV[1];
    const float dz = (pv.detS[2] + float(u) * pv.detU[2]) + float(v) * pv.detV[2];
    const float sx = pv.src[0], sy = pv.src[1], sz = pv.src[2];
    const float s0 = pick(ax.p0, sx, sy, sz), s1 = pick(ax.p1, sx, sy, sz), s2 = pick(ax.p2, sx, sy, sz);
    const float d0 = pick(ax.p0, dx, dy, dz), d1 = pick(ax.p1, dx, dy, dz), d2 = pick(ax.p2, dx, dy, dz);
    const float den = s0 - d0;
    if (den == 0.f) return false;
    r.a1 = (s1 - d1) / den;
    r.a2 = (s2 - d2) / den;
    r.b1 = s1 - r.a1 * s0;
    r.b2 = s2 - r.a2 * s0;
    const float t1 = r.a1 * ax.v1, t2 = r.a2 * ax.v2;
    r.L = sqrtf(ax.v0 * ax.v0 + t1 * t1 + t2 * t2);
    return true;
}

// centred main-axis coordinate of slice s
__device__ __forceinline__ float joseph_c0(int s, int n0)
{
#pragma clang fp contract(off)
    return float(s) - 0.5f * float(n0 - 1);
}

// one minor-axis sample position (index space, texel k at k) of the line
// c = a c0 + b
__device__ __forceinline__ float joseph_minor(float a, float b, float c0, int n)
{
#pragma clang fp contract(off)
    return (a * c0 + b) + 0.5f * float(n - 1);
}

__device__ __forceinline__ void siddon_ray_geom(const SiddonViewDev& sv, int u, int v, float* src, float* ray)
{
#pragma clang fp contract(off)
    for (int k = 0; k < 3; ++k) {
        src[k] = sv.src[k];
        ray[k] = (sv.detS[k] + float(u) * sv.detU[k] + float(v) * sv.detV[k]) - sv.src[k];
    }
}

// the same in FP64: pixel minus source
__device__ __forceinline__ void siddon_ray_geom(const SiddonViewDev& sv, int u, int v, double* ray)
{
    for (int k = 0; k < 3; ++k)
        ray[k] = (double(sv.detS[k]) + u * double(sv.detU[k]) + v * double(sv.detV[k])) - double(sv.src[k]);
}

// A ray that moves `along` cells of its main axis, of n0, and `across` cells of
// another, of n, in the same time stays in one cell layer of that axis if it moves
// no further across the volume than FP32 resolves there.  If the source lies on a
// plane between cells (SiddonViewDev::plane) the layer is the upper one.  The
// projection and the transposes have to agree on that: the ray's whole
// contribution is at stake, not a rounding of it.
__device__ __forceinline__ bool siddon_stays(double across, int n, double along, int n0)
{
    return fabs(across) * n0 <= fabs(along) * (n * 0x1p-22);
}

// whether a ray lies in an upper face of the volume, and so in no cell
__device__ __forceinline__ bool siddon_in_upper_face(const SiddonViewDev& sv, const VolumeGeom& g, int u, int v)
{
    const int n[3] = { g.nx, g.ny, g.nz };
    if (sv.plane[0] != n[0] && sv.plane[1] != n[1] && sv.plane[2] != n[2]) return false;
    double r[3];
    siddon_ray_geom(sv, u, v, r);
    r[0] /= g.vx;
    r[1] /= g.vy;
    r[2] /= g.vz;
    int m = fabs(r[0]) >= fabs(r[1]) ? 0 : 1;
    if (fabs(r[2]) > fabs(m == 0 ? r[0] : r[1])) m = 2;
    const double along = m == 0 ? r[0] : m == 1 ? r[1] : r[2];
    const int n0 = m == 0 ? n[0] : m == 1 ? n[1] : n[2];
    bool in = false;
    for (int k = 0; k < 3; ++k) in = in || (k != m && sv.plane[k] == n[k] && siddon_stays(r[k], n[k], along, n0));
    return in;
}

struct Box {
    float lo[3], hi[3];
};

__device__ __forceinline__ Box volume_box(const VolumeGeom& g)
{
    Box b;
    b.lo[0] = g.ox - 0.5f * g.vx; b.hi[0] = g.ox + (float(g.nx) - 0.5f) * g.vx;
    b.lo[1] = g.oy - 0.5f * g.vy; b.hi[1] = g.oy + (float(g.ny) - 0.5f) * g.vy;
    b.lo[2] = g.oz - 0.5f * g.vz; b.hi[2] = g.oz + (float(g.nz) - 0.5f) * g.vz;
    return b;
}

// one slab of the box clip: narrows [t0, t1] to lo <= s + t r <= hi; a ray
// parallel to the slab and outside it misses
__device__ __forceinline__ bool slab_clip(float s, float r, float lo, float hi, float& t0, float& t1)
{
    if (fabsf(r) > 1e-8f) {
        float ta = (lo - s) / r, tb = (hi - s) / r;
        if (ta > tb) { const float t = ta; ta = tb; tb = t; }
        t0 = fmaxf(t0, ta);
        t1 = fminf(t1, tb);
        return true;
    }
    return !(s < lo || s > hi);
}

// parametric segment [t0, t1] of src + t ray inside the box, clipped to [0, 1]
__device__ __forceinline__ bool clip_ray(const float* src, const float* ray, const float* lo,
    const float* hi, float& t0, float& t1)
{
    t0 = 0.f;
    t1 = 1.f;
    for (int k = 0; k < 3; ++k)
        if (!slab_clip(src[k], ray[k], lo[k], hi[k], t0, t1)) return false;
    return t0 < t1;
}

// t-interval of the walk inside cell c of one axis: the forward walk's own
// plane crossings (plane - src) * (1 / ray); a ray parallel to the axis stays
// in the cell its source coordinate lies in
__device__ __forceinline__ void cell_interval(float s, float r, float lo, float vox, int c, int n,
    float& ta, float& tb)
{
    if (fabsf(r) > 1e-8f) {
        const float rc = 1.f / r;
        const float t0 = (lo + float(c) * vox - s) * rc, t1 = (lo + float(c + 1) * vox - s) * rc;
        ta = fmaxf(ta, fminf(t0, t1));
        tb = fminf(tb, fmaxf(t0, t1));
    } else if (min(n - 1, max(0, int(floorf((s - lo) / vox)))) != c) {
        tb = -3.0e38f;
    }
}

// world projective map (u or v numerator row r, denominator row d) of a point
__device__ __forceinline__ float proj_coord(const float* c, int row, float x, float y, float z, float rd)
{
    return (c[row] * x + c[row + 1] * y + c[row + 2] * z + c[row + 3]) * rd;
}

}  // namespace
}  // namespace yk
