// Transposes of the Joseph and Siddon projections for views of any orientation
// with main axis X or Y (tilted detectors, lifted sources), as deterministic
// gathers for gfx950.
//
// Joseph: a ray (u, v) of a view leaves the source s towards the pixel
// d(u, v), in volume-centred voxel units with components 0 (main axis), 1
// (first minor axis) and 2 (z).  With D = d0 - s0 and e_k = d_k - s_k, all
// linear in (u, v), its offset on minor axis k from voxel (c0, c1, c2), where
// it crosses the voxel's main-axis plane, is N_k / D with
//   N_k = (s_k - c_k) D + (c0 - s0) e_k,
// linear in (u, v) too, and it adds
//   p L max(0, 1 - |N1 / D|) max(0, 1 - |N2 / D|)
//     = q max(0, |D| - |N1|) max(0, |D| - |N2|),   q = p L / D^2.
// A candidate therefore costs ten instructions for two voxels and one 4-byte
// table value, where evaluating its line took 24 bytes of table and a floor /
// compare chain for each.  N_k at a reference pixel near the voxel is formed in
// FP64 (its terms are a thousand times the result) and carried to the
// candidates in FP32 steps.
//
// Siddon: the segment of a ray in a voxel lies between its crossings of the
// voxel's six planes, at (plane - src) * (main / minor component) along the main
// axis; the quotients come from a table of the view's rays (12 bytes with
// p |ray / main|) instead of three divisions per candidate.
//
// 256^3 x 360 views of 512 x 384, detector tilted: Joseph 118.7 -> 15.9 ms,
// Siddon 139.7 -> 20.9 ms against one thread per voxel with every candidate's
// line evaluated; then, for Siddon, medians in place of sorted intervals -> 16.5
// and quotients along the main axis (12 bytes and 14 instructions a candidate
// for 16 and 16) -> 16.1.  64^3 x 60 views of 128 x 96: 1.15 -> 0.09 and 1.75 ->
// 0.11 ms.  Untilted views have forms of their own where they are faster
// (kernels_column.hip, siddon_flat_gather).
// Bound: VALU issue (Joseph: 324 instructions a voxel pair and view, of which 218
// weigh its 5.4 rows of 4 candidates; the texture addressers are 67 % busy) or the
// addressers (Siddon: six 12-byte loads for 84 instructions, 95 % busy; untilted 84
// %); profiles/projectors_counters.txt.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ray_geometry.hpp"
#include "yk_internal.hpp"

namespace yk {
namespace {

typedef float float4a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float float3a4 __attribute__((ext_vector_type(3), aligned(4)));
typedef float float2a4 __attribute__((ext_vector_type(2), aligned(4)));

// clamp to [0, 1]: the output modifier of the instruction that forms x
__device__ __forceinline__ float sat(float x) { return __builtin_amdgcn_fmed3f(x, 0.f, 1.f); }

__global__ void gather_clear_kernel(int* __restrict__ flag) { *flag = 0; }

// q of every ray, [view][v][pitch], zero in the pitch - nu columns closing each
// row and the kGatherPadRows rows closing each view.  A value that is not finite raises *flag: a gather then skips, rather
// than weighs with zero, the candidates that do not meet a voxel.
__global__ void __launch_bounds__(256)
joseph_gather_table_kernel(const float* __restrict__ proj, const ProjViewDev* __restrict__ views,
    const GatherViewDev* __restrict__ gviews, VolumeGeom g, int nu, int nv, int pitch, float* __restrict__ q,
    int* __restrict__ flag)
{
    const int u = blockIdx.x * 64 + threadIdx.x;
    const int v = blockIdx.y * 4 + threadIdx.y, i = blockIdx.z;
    const int rows = nv + kGatherPadRows;
    if (u >= pitch || v >= rows) return;
    float w = 0.f;
    if (u < nu && v < nv) {
        const ProjViewDev pv = views[i];
        const AxisInfo ax = axis_info(pv.axis, g);
        JRay r;
        if (joseph_ray(pv, ax, u, v, r)) {
            const float d = ((pick(ax.p0, pv.detS[0], pv.detS[1], pv.detS[2]) - pick(ax.p0, pv.src[0], pv.src[1], pv.src[2])) +
                float(u) * pick(ax.p0, pv.detU[0], pv.detU[1], pv.detU[2]) +
                float(v) * pick(ax.p0, pv.detV[0], pv.detV[1], pv.detV[2])) * gviews[i].scale;
            w = proj[((size_t)i * nv + v) * nu + u] * r.L / (d * d);
        }
        if (!(fabsf(w) <= 3.4e38f)) atomicOr(flag, 1);
    }
    q[((size_t)i * rows + v) * pitch + u] = w;
}

// (main / first minor, main / z component, p |ray / main|) of every ray, same
// layout; a minor component the ray does not move along (siddon_stays) has a
// quotient so large that its cell either bounds nothing or leaves no segment,
// with the main component's sign: the cell's upper plane is then always the
// farther one along the ray
__global__ void __launch_bounds__(256)
siddon_gather_table_kernel(const float* __restrict__ proj, const SiddonViewDev* __restrict__ views,
    const GatherViewDev* __restrict__ gviews, VolumeGeom g, int nu, int nv, int pitch, float* __restrict__ q,
    int* __restrict__ flag)
{
    const int u = blockIdx.x * 64 + threadIdx.x;
    const int v = blockIdx.y * 4 + threadIdx.y, i = blockIdx.z;
    const int rows = nv + kGatherPadRows;
    if (u >= pitch || v >= rows) return;
    float r1 = 0.f, r2 = 0.f, w = 0.f;
    if (u < nu && v < nv) {
        double r[3];
        siddon_ray_geom(views[i], u, v, r);
        const bool xmain = gviews[i].axis == 0;
        const int n0 = xmain ? g.nx : g.ny, n1 = xmain ? g.ny : g.nx;
        const double along = (xmain ? r[0] : r[1]) * (xmain ? g.vy * g.vz : g.vx * g.vz);  // (cells, times vx vy vz)
        const float ray[3] = { float(r[0]), float(r[1]), float(r[2]) };
        const float m0 = xmain ? ray[0] : ray[1], m1 = xmain ? ray[1] : ray[0];
        const float far = copysignf(1e30f, m0);
        r1 = siddon_stays((xmain ? r[1] : r[0]) * (xmain ? g.vx * g.vz : g.vy * g.vz), n1, along, n0) ? far : m0 / m1;
        r2 = siddon_stays(r[2] * (g.vx * g.vy), g.nz, along, n0) ? far : m0 / ray[2];
        w = proj[((size_t)i * nv + v) * nu + u] * (sqrtf(ray[0] * ray[0] + ray[1] * ray[1] + ray[2] * ray[2]) / fabsf(m0));
        if (!(fabsf(w) <= 3.4e38f)) atomicOr(flag, 1);
    }
    float* dst = q + 3 * (((size_t)i * rows + v) * pitch + u);
    dst[0] = r1;
    dst[1] = r2;
    dst[2] = w;
}

// The same of views whose detector rows and columns lie along the main axes'
// plane and z (separable, no z in a row's step): a ray's x and y do not depend
// on v, nor its z on u, so the reciprocals are one entry a column, ru [view]
// [pitch] (1 / x, 1 / y), and one a row, rv [view][nv + kGatherPadRows]; q is
// p |ray| alone.
__global__ void __launch_bounds__(256)
siddon_flat_table_kernel(const float* __restrict__ proj, const SiddonViewDev* __restrict__ views, VolumeGeom g, int nu, int nv,
    int pitch, float* __restrict__ q, float2* __restrict__ ru, float* __restrict__ rv, int* __restrict__ flag)
{
    const int u = blockIdx.x * 64 + threadIdx.x;
    const int v = blockIdx.y * 4 + threadIdx.y, i = blockIdx.z;
    const int rows = nv + kGatherPadRows;
    if (u >= pitch || v >= rows) return;
    float src[3], ray[3];
    siddon_ray_geom(views[i], u, v, src, ray);
    float w = 0.f;
    if (u < nu && v < nv) {
        w = proj[((size_t)i * nv + v) * nu + u] * sqrtf(ray[0] * ray[0] + ray[1] * ray[1] + ray[2] * ray[2]);
        if (!(fabsf(w) <= 3.4e38f)) atomicOr(flag, 1);
    }
    q[((size_t)i * rows + v) * pitch + u] = w;
    if (u > 0 && v > 0) return;
    double r[3];
    siddon_ray_geom(views[i], u, v, r);
    // (cells, times vx vy vz)
    const double cx = r[0] * (g.vy * g.vz), cy = r[1] * (g.vx * g.vz), cz = r[2] * (g.vx * g.vy);
    const bool xmain = fabs(cx) >= fabs(cy);
    auto quotient = [](bool stays, double r) { return stays || r == 0.0 ? 1e30f : 1.f / float(r); };
    if (v == 0)
        ru[(size_t)i * pitch + u] = make_float2(quotient(!xmain && siddon_stays(cx, g.nx, cy, g.ny), r[0]),
            quotient(xmain && siddon_stays(cy, g.ny, cx, g.nx), r[1]));
    if (u == 0) rv[(size_t)i * rows + v] = quotient(siddon_stays(cz, g.nz, xmain ? cx : cy, xmain ? g.nx : g.ny), r[2]);
}

// Where the candidates of a lane's run of ZR voxels along z lie on one view.
// A lane walks its run two voxels at a time: a pair shares the rows both see
// (for Joseph 5.1 instead of 2 x 3.4 at a magnified voxel of 1.7 pixels).  The
// candidate box is the projection of the pair's support with 0.05 px of margin
// against FP32 rounding; weights vanish by themselves outside the support, so
// the box only has to contain it and is walked in chunks of a fixed width.
// kHalf*: half extents of the support, in voxels (main axis, first minor, z).
template <int ZR>
struct CandidateBox {
    float u0, v0, d0;  // numerators of u and v, and depth, at (x, y, 0)
    float u_z, v_z, a_z;
    float um, vm;      // the middle of the run
    float v_zd;        // v a voxel along z, of views whose depth does not vary along z
    float hu, hv;      // half widths of a pair's box anywhere in the run

    __device__ __forceinline__ CandidateBox(const GatherViewDev& r, int x, int y, int z0, float h_main, float h_1,
        float h_z)
    {
        const bool xmain = r.axis == 0;
        const float fx = float(x), fy = float(y);
        u0 = fmaf(r.mu[0], fx, fmaf(r.mu[1], fy, r.mu[3]));
        v0 = fmaf(r.mv[0], fx, fmaf(r.mv[1], fy, r.mv[3]));
        d0 = fmaf(r.md[0], fx, fmaf(r.md[1], fy, r.md[3]));
        u_z = r.mu[2], v_z = r.mv[2], a_z = r.md[2];
        const float a_main = xmain ? r.md[0] : r.md[1], a_1 = xmain ? r.md[1] : r.md[0];
        const float u_main = xmain ? r.mu[0] : r.mu[1], u_1 = xmain ? r.mu[1] : r.mu[0];
        const float v_main = xmain ? r.mv[0] : r.mv[1], v_1 = xmain ? r.mv[1] : r.mv[0];
        const float dhalf = h_main * fabsf(a_main) + h_1 * fabsf(a_1) + h_z * fabsf(a_z);
        // A corner of a support departs from its centre by at most sum h
        // |numerator slope - f depth slope| / (least depth of the support), f
        // = u or v at the centre, which over the run departs from the middle's
        // by at most su, sv (the same bound along z).  Every depth here is
        // positive (projector.cpp, depth_range).
        const float zm = float(z0) + 0.5f * float(ZR - 1);
        const float dm = fmaf(a_z, zm, d0);
        const float rm = __builtin_amdgcn_rcpf(dm);
        const float rb = __builtin_amdgcn_rcpf(dm - fmaf(0.5f * float(ZR), fabsf(a_z), dhalf));
        um = fmaf(u_z, zm, u0) * rm;
        vm = fmaf(v_z, zm, v0) * rm;
        v_zd = v_z * rm;
        const float ku = fabsf(fmaf(-um, a_z, u_z)) * rb, kv = fabsf(fmaf(-vm, a_z, v_z)) * rb;
        const float su = 0.5f * float(ZR) * ku, sv = 0.5f * float(ZR) * kv;
        hu = fmaf(h_z, ku, fmaf(h_1, fabsf(fmaf(-um, a_1, u_1)) * rb, fmaf(su * dhalf, rb, 0.05f)));
        hv = fmaf(h_z, kv, fmaf(h_1, fabsf(fmaf(-vm, a_1, v_1)) * rb, fmaf(sv * dhalf, rb, 0.05f)));
        if (h_main > 0.f) {
            hu = fmaf(h_main, fabsf(fmaf(-um, a_main, u_main)) * rb, hu);
            hv = fmaf(h_main, fabsf(fmaf(-vm, a_main, v_main)) * rb, hv);
        }
    }

    // pixel ranges of the pair whose lower voxel is z; false when empty
    __device__ __forceinline__ bool pair(int z, int nu, int nv, int& ulo, int& uhi, int& vlo, int& vhi) const
    {
        const float zc = float(z) + 0.5f;
        const float rd = __builtin_amdgcn_rcpf(fmaf(a_z, zc, d0));
        const float uc = fmaf(u_z, zc, u0) * rd, vc = fmaf(v_z, zc, v0) * rd;
        ulo = int(fmaxf(0.f, ceilf(uc - hu))), uhi = int(fminf(float(nu - 1), floorf(uc + hu)));
        vlo = int(fmaxf(0.f, ceilf(vc - hv))), vhi = int(fminf(float(nv - 1), floorf(vc + hv)));
        return ulo <= uhi && vlo <= vhi;
    }
};

// A lane holds one (x, y), a workgroup 16 x 16, so the lanes of a wave read
// neighbouring pixels of a few rows.
template <int ZR, bool SAFE>
__device__ __forceinline__ void joseph_gather(const float* __restrict__ q, const GatherViewDev* __restrict__ views,
    const VolumeGeom& g, int nu, int nv, int pitch, int count, int x, int y, int z0, float (&acc)[ZR])
{
    constexpr int kWidth = 4, kRows = 3;  // 2 or 1 rows a chunk measured 0-10 % slower
    const double zc0 = double(z0) - 0.5 * double(g.nz - 1);
#pragma unroll 1
    for (int i = 0; i < count; ++i) {
        const GatherViewDev& r = views[i];
        const bool xmain = r.axis == 0;
        const float* qi = q + (size_t)i * (nv + kGatherPadRows) * pitch;
        const CandidateBox<ZR> box(r, x, y, z0, 0.f, 1.f, 1.5f);
        const int ur = int(__builtin_amdgcn_fmed3f(box.um, 0.f, float(nu)));
        const int vr = int(__builtin_amdgcn_fmed3f(box.vm, 0.f, float(nv)));
        const double c0 = double(xmain ? x : y) - 0.5 * double((xmain ? g.nx : g.ny) - 1);
        const double c1 = double(xmain ? y : x) - 0.5 * double((xmain ? g.ny : g.nx) - 1);
        const double k0 = c0 - r.src[0], a1 = r.src[1] - c1, a2 = r.src[2] - zc0;
        const double dr = fma(double(vr), r.d[2], fma(double(ur), r.d[1], r.d[0]));
        const double e1r = fma(double(vr), r.e1[2], fma(double(ur), r.e1[1], r.e1[0]));
        const double e2r = fma(double(vr), r.e2[2], fma(double(ur), r.e2[1], r.e2[0]));
        const float n1r = float(fma(a1, dr, k0 * e1r)), n2r = float(fma(a2, dr, k0 * e2r)), drf = float(dr);
        const float k0f = float(k0), a1f = float(a1), a2f = float(a2);
        const float du = float(r.d[1]), dv = float(r.d[2]);
        const float e2u = float(r.e2[1]), e2v = float(r.e2[2]);
        const float n1u = fmaf(a1f, du, k0f * float(r.e1[1])), n1v = fmaf(a1f, dv, k0f * float(r.e1[2]));
#pragma unroll
        for (int p = 0; p < ZR; p += 2) {
            int ulo, uhi, vlo, vhi;
            if (!box.pair(z0 + p, nu, nv, ulo, uhi, vlo, vhi)) continue;
            const float fu = float(ulo - ur), fv = float(vlo - vr);
            float d_row = fmaf(fu, du, fmaf(fv, dv, drf));
            float n1_row = fmaf(fu, n1u, fmaf(fv, n1v, n1r));
            const float n2u = fmaf(a2f - float(p), du, k0f * e2u), n2v = fmaf(a2f - float(p), dv, k0f * e2v);
            float n2_row = fmaf(fu, n2u, fmaf(fv, n2v, fmaf(-float(p), drf, n2r)));
            unsigned row = unsigned(vlo) * unsigned(pitch);
#pragma unroll 1
            for (int v = vlo; v <= vhi; v += kRows) {
                float d_u = d_row, n1_u = n1_row, n2_u = n2_row;
#pragma unroll 1
                for (int u = ulo; u <= uhi; u += kWidth) {
                    // every load of the chunk is issued before any is consumed
                    float4a4 w[kRows];
#pragma unroll
                    for (int j = 0; j < kRows; ++j)
                        w[j] = *reinterpret_cast<const float4a4*>(qi + (row + unsigned(j * pitch + u)));
#pragma unroll
                    for (int j = 0; j < kRows; ++j) {
                        float d = fmaf(float(j), dv, d_u), n1 = fmaf(float(j), n1v, n1_u), n2 = fmaf(float(j), n2v, n2_u);
#pragma unroll
                        for (int k = 0; k < kWidth; ++k) {
                            const float w1 = sat(fabsf(d) - fabsf(n1));
                            const float wa = sat(fabsf(d) - fabsf(n2)), wb = sat(fabsf(d) - fabsf(n2 - d));
                            const float t = w1 * w[j][k];
                            if (!SAFE || (w1 > 0.f && wa > 0.f)) acc[p] = fmaf(t, wa, acc[p]);
                            if (!SAFE || (w1 > 0.f && wb > 0.f)) acc[p + 1] = fmaf(t, wb, acc[p + 1]);
                            d += du;
                            n1 += n1u;
                            n2 += n2u;
                        }
                    }
                    d_u = fmaf(float(kWidth), du, d_u);
                    n1_u = fmaf(float(kWidth), n1u, n1_u);
                    n2_u = fmaf(float(kWidth), n2u, n2_u);
                }
                row += unsigned(kRows * pitch);
                d_row = fmaf(float(kRows), dv, d_row);
                n1_row = fmaf(float(kRows), n1v, n1_row);
                n2_row = fmaf(float(kRows), n2v, n2_row);
            }
        }
    }
}

// offset of plane c between cells from the source (SiddonViewDev::on_plane):
// exactly zero on the source's own plane
__device__ __forceinline__ float plane_offset(float lo, float vox, int c, float s) { return fmaf(float(c), vox, lo) - s; }

template <int ZR, bool SAFE>
__device__ __forceinline__ void siddon_gather(const float* __restrict__ q, const GatherViewDev* __restrict__ views,
    const SiddonViewDev* __restrict__ sviews, const VolumeGeom& g, int nu, int nv, int pitch, int count, int x, int y,
    int z0, float (&acc)[ZR])
{
    // 1-4 pixels x 1-4 rows a chunk measured 20.5-24.7 ms at 256^3 x 360 views,
    // this one 20.9 but 5-10 % ahead of the others at 128^3 and 64^3
    constexpr int kWidth = 3, kRows = 2;
    const float lox = g.ox - 0.5f * g.vx, loy = g.oy - 0.5f * g.vy, loz = g.oz - 0.5f * g.vz;
#pragma unroll 1
    for (int i = 0; i < count; ++i) {
        const float* qi = q + 3 * ((size_t)i * (nv + kGatherPadRows) * pitch);
        const CandidateBox<ZR> box(views[i], x, y, z0, 0.5f, 0.5f, 1.f);
        const SiddonViewDev& sv = sviews[i];
        const float x0 = plane_offset(lox, g.vx, x, sv.on_plane[0]);
        const float x1 = plane_offset(lox, g.vx, x + 1, sv.on_plane[0]);
        const float y0 = plane_offset(loy, g.vy, y, sv.on_plane[1]);
        const float y1 = plane_offset(loy, g.vy, y + 1, sv.on_plane[1]);
        const bool xmain = views[i].axis == 0;
        const float m0 = xmain ? x0 : y0, m1 = xmain ? x1 : y1, n0 = xmain ? y0 : x0, n1 = xmain ? y1 : x1;
#pragma unroll
        for (int p = 0; p < ZR; p += 2) {
            int ulo, uhi, vlo, vhi;
            if (!box.pair(z0 + p, nu, nv, ulo, uhi, vlo, vhi)) continue;
            const float za = plane_offset(loz, g.vz, z0 + p, sv.on_plane[2]);
            const float zb = plane_offset(loz, g.vz, z0 + p + 1, sv.on_plane[2]);
            const float zc = plane_offset(loz, g.vz, z0 + p + 2, sv.on_plane[2]);
            unsigned row = unsigned(vlo) * unsigned(pitch);
#pragma unroll 1
            for (int v = vlo; v <= vhi; v += kRows) {
#pragma unroll 1
                for (int u = ulo; u <= uhi; u += kWidth) {
                    float3a4 w[kRows][kWidth];
#pragma unroll
                    for (int j = 0; j < kRows; ++j)
#pragma unroll
                        for (int k = 0; k < kWidth; ++k)
                            w[j][k] = *reinterpret_cast<const float3a4*>(qi + 3u * (row + unsigned(j * pitch + u + k)));
#pragma unroll
                    for (int j = 0; j < kRows; ++j)
#pragma unroll
                        for (int k = 0; k < kWidth; ++k) {
                            const float3a4 c = w[j][k];
                            // Along the main axis the ray is between the voxel's
                            // planes from m0 to m1; a median moves the crossings of
                            // the minor planes into that interval and those of the z
                            // planes into what is left (empty: onto one point), with
                            // no interval sorted.  25 -> 14 instructions a candidate
                            // against sorted ends of three axes.
                            const float na = __builtin_amdgcn_fmed3f(n0 * c.x, m0, m1), nb = __builtin_amdgcn_fmed3f(n1 * c.x, m0, m1);
                            const float ta = __builtin_amdgcn_fmed3f(za * c.y, na, nb);
                            const float tb = __builtin_amdgcn_fmed3f(zb * c.y, na, nb);
                            const float tc = __builtin_amdgcn_fmed3f(zc * c.y, na, nb);
                            const float sa = fabsf(tb - ta), sb = fabsf(tc - tb);
                            if (!SAFE || sa > 0.f) acc[p] = fmaf(sa, c.z, acc[p]);
                            if (!SAFE || sb > 0.f) acc[p + 1] = fmaf(sb, c.z, acc[p + 1]);
                        }
                }
                row += unsigned(kRows * pitch);
            }
        }
    }
}

// Views of siddon_flat_table_kernel.  Depth, the candidate columns and the part
// of each column's rays over the voxel column's x and y planes hold for the
// whole run, and a row's z planes for all its candidates, so a candidate takes 7
// instructions and 4 bytes where siddon_gather takes 14 and 12.  Against 16
// and 16: 256^3 x 360
// views of 512 x 384 17.2 -> 10.4 ms, 128^3 x 120 891 -> 570 us, 64^3 x 60 116
// -> 102.  (Pixels x rows a chunk at 256^3: 3 x 1 12.9 ms, 3 x 3 11.2, 2 x 2
// 22.3, 4 x 2 10.9.)
// ENDS: a ray ends at its pixel, t = 1, inside the volume of some view (5 % on
// the others).
template <int ZR, bool SAFE, bool ENDS>
__device__ __forceinline__ void siddon_flat_gather(const float* __restrict__ q, const float2* __restrict__ ru,
    const float* __restrict__ rv, const GatherViewDev* __restrict__ views, const SiddonViewDev* __restrict__ sviews,
    const VolumeGeom& g, int nu, int nv, int pitch, int count, int x, int y, int z0, float (&acc)[ZR])
{
    constexpr int kWidth = 3, kRows = 2;
    const float lox = g.ox - 0.5f * g.vx, loy = g.oy - 0.5f * g.vy, loz = g.oz - 0.5f * g.vz;
#pragma unroll 1
    for (int i = 0; i < count; ++i) {
        const size_t rows = size_t(i) * (nv + kGatherPadRows);
        const float* qi = q + rows * pitch;
        const float* rvi = rv + rows;
        const CandidateBox<ZR> box(views[i], x, y, z0, 0.5f, 0.5f, 1.f);
        const SiddonViewDev& sv = sviews[i];
        const float x0 = plane_offset(lox, g.vx, x, sv.on_plane[0]);
        const float x1 = plane_offset(lox, g.vx, x + 1, sv.on_plane[0]);
        const float y0 = plane_offset(loy, g.vy, y, sv.on_plane[1]);
        const float y1 = plane_offset(loy, g.vy, y + 1, sv.on_plane[1]);
        const int ulo = int(fmaxf(0.f, ceilf(box.um - box.hu))), uhi = int(fminf(float(nu - 1), floorf(box.um + box.hu)));
#pragma unroll 1
        for (int u = ulo; u <= uhi; u += kWidth) {
            float ya[kWidth], yb[kWidth];
#pragma unroll
            for (int k = 0; k < kWidth; ++k) {
                const float2 c = ru[(size_t)i * pitch + (u + k)];
                const float tx0 = x0 * c.x, tx1 = x1 * c.x;
                ya[k] = __builtin_amdgcn_fmed3f(y0 * c.y, tx0, tx1);
                yb[k] = __builtin_amdgcn_fmed3f(y1 * c.y, tx0, tx1);
                if constexpr (ENDS) {
                    ya[k] = fminf(ya[k], 1.f);
                    yb[k] = fminf(yb[k], 1.f);
                }
            }
#pragma unroll
            for (int p = 0; p < ZR; p += 2) {
                const float vc = fmaf(box.v_zd, float(p) + 0.5f - 0.5f * float(ZR - 1), box.vm);
                const int vlo = int(fmaxf(0.f, ceilf(vc - box.hv))), vhi = int(fminf(float(nv - 1), floorf(vc + box.hv)));
                const float za = plane_offset(loz, g.vz, z0 + p, sv.on_plane[2]);
                const float zb = plane_offset(loz, g.vz, z0 + p + 1, sv.on_plane[2]);
                const float zc = plane_offset(loz, g.vz, z0 + p + 2, sv.on_plane[2]);
                unsigned row = unsigned(vlo) * unsigned(pitch) + unsigned(u);
#pragma unroll 1
                for (int v = vlo; v <= vhi; v += kRows) {
                    float3a4 w[kRows];
#pragma unroll
                    for (int j = 0; j < kRows; ++j) w[j] = *reinterpret_cast<const float3a4*>(qi + (row + unsigned(j * pitch)));
                    const float2a4 r = *reinterpret_cast<const float2a4*>(rvi + unsigned(v));
#pragma unroll
                    for (int j = 0; j < kRows; ++j) {
                        const float za_t = za * r[j], zb_t = zb * r[j], zc_t = zc * r[j];
#pragma unroll
                        for (int k = 0; k < kWidth; ++k) {
                            const float ta = __builtin_amdgcn_fmed3f(za_t, ya[k], yb[k]);
                            const float tb = __builtin_amdgcn_fmed3f(zb_t, ya[k], yb[k]);
                            const float tc = __builtin_amdgcn_fmed3f(zc_t, ya[k], yb[k]);
                            const float sa = fabsf(tb - ta), sb = fabsf(tc - tb);
                            if (!SAFE || sa > 0.f) acc[p] = fmaf(sa, w[j][k], acc[p]);
                            if (!SAFE || sb > 0.f) acc[p + 1] = fmaf(sb, w[j][k], acc[p + 1]);
                        }
                    }
                    row += unsigned(kRows * pitch);
                }
            }
        }
    }
}

template <int MODEL, int ZR>
__global__ void __launch_bounds__(256)
gather_transpose_kernel(const void* __restrict__ q, const float2* __restrict__ ru, const float* __restrict__ rv,
    float* __restrict__ volume, const GatherViewDev* __restrict__ views, const SiddonViewDev* __restrict__ sviews,
    const int* __restrict__ flag, VolumeGeom g, int nu, int nv, int pitch, int count, int accumulate)
{
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    const int z0 = blockIdx.z * ZR;
    if (x >= g.nx || y >= g.ny) return;
    float acc[ZR];
#pragma unroll
    for (int k = 0; k < ZR; ++k) acc[k] = 0.f;
    const bool plain = __builtin_amdgcn_readfirstlane(*flag) == 0;
    if constexpr (MODEL == kGatherSiddonFlat || MODEL == kGatherSiddonFlatEnds) {
        constexpr bool kEnds = MODEL == kGatherSiddonFlatEnds;
        const float* t = static_cast<const float*>(q);
        if (plain) siddon_flat_gather<ZR, false, kEnds>(t, ru, rv, views, sviews, g, nu, nv, pitch, count, x, y, z0, acc);
        else siddon_flat_gather<ZR, true, kEnds>(t, ru, rv, views, sviews, g, nu, nv, pitch, count, x, y, z0, acc);
    } else if constexpr (MODEL == kGatherSiddon) {
        const float* t = static_cast<const float*>(q);
        if (plain) siddon_gather<ZR, false>(t, views, sviews, g, nu, nv, pitch, count, x, y, z0, acc);
        else siddon_gather<ZR, true>(t, views, sviews, g, nu, nv, pitch, count, x, y, z0, acc);
    } else {
        const float* t = static_cast<const float*>(q);
        if (plain) joseph_gather<ZR, false>(t, views, g, nu, nv, pitch, count, x, y, z0, acc);
        else joseph_gather<ZR, true>(t, views, g, nu, nv, pitch, count, x, y, z0, acc);
    }
    const size_t plane = (size_t)g.nx * g.ny;
#pragma unroll
    for (int k = 0; k < ZR; ++k) {
        if (z0 + k >= g.nz) break;
        float* dst = volume + (size_t)(z0 + k) * plane + (size_t)y * g.nx + x;
        *dst = accumulate ? *dst + acc[k] : acc[k];
    }
}

template <int MODEL, int ZR>
void launch_run(const GatherLaunch& p, hipStream_t s)
{
    const VolumeGeom& g = p.vol;
    dim3 grid((g.nx + 15) / 16, (g.ny + 15) / 16, (g.nz + ZR - 1) / ZR);
    hipLaunchKernelGGL((gather_transpose_kernel<MODEL, ZR>), grid, dim3(256), 0, s, p.q, p.ru, p.rv, p.volume, p.gviews, p.sviews,
        p.flag, g, p.nu, p.nv, p.pitch, p.count, p.accumulate);
    YK_HIP(hipGetLastError());
}

template <int MODEL>
void launch_gather(const GatherLaunch& p, hipStream_t s)
{
    const VolumeGeom& g = p.vol;
    const long wide = long((g.nx + 15) / 16) * ((g.ny + 15) / 16) * ((g.nz + kGatherRun - 1) / kGatherRun);
    // (the longer run shares a view's setup among more voxels, the shorter
    // one has four times the workgroups: at 60 views and 128^3 = 1024
    // workgroups both take 432 us, at 160^3 724 against 811, at 112^3 346
    // against 304, at 64^3 236 against 96)
    if (wide >= 1024) launch_run<MODEL, kGatherRun>(p, s);
    else launch_run<MODEL, 2>(p, s);
}

}  // namespace

void launch_gather_transpose(const GatherLaunch& p, hipStream_t s)
{
    hipLaunchKernelGGL(gather_clear_kernel, dim3(1), dim3(1), 0, s, p.flag);
    // (64 x 4 rays a workgroup: 256 rays of one row left half of them idle at a
    // pitch of 260; CGLS at 128^3 x 120 views of 256 x 192 5.84 -> 5.76 ms)
    dim3 tb(64, 4), tg((p.pitch + 63) / 64, (p.nv + kGatherPadRows + 3) / 4, p.count);
    if (p.model == kGatherSiddonFlat || p.model == kGatherSiddonFlatEnds) {
        hipLaunchKernelGGL(siddon_flat_table_kernel, tg, tb, 0, s, p.proj, p.sviews, p.vol, p.nu, p.nv, p.pitch, p.q, p.ru,
            p.rv, p.flag);
        if (p.model == kGatherSiddonFlatEnds) launch_gather<kGatherSiddonFlatEnds>(p, s);
        else launch_gather<kGatherSiddonFlat>(p, s);
    } else if (p.model == kGatherSiddon) {
        hipLaunchKernelGGL(siddon_gather_table_kernel, tg, tb, 0, s, p.proj, p.sviews, p.gviews, p.vol, p.nu,
            p.nv, p.pitch, p.q, p.flag);
        launch_gather<kGatherSiddon>(p, s);
    } else {
        hipLaunchKernelGGL(joseph_gather_table_kernel, tg, tb, 0, s, p.proj, p.views, p.gviews, p.vol, p.nu, p.nv,
            p.pitch, p.q, p.flag);
        launch_gather<kGatherJoseph>(p, s);
    }
}

}  // namespace yk
