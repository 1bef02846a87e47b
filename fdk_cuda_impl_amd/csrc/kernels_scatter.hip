// Transposes of untilted views (main axis X or Y, detector columns along z) by
// scattering, for gfx950: each lane holds an (x, y) column of voxels in LDS and
// walks the rays of the detector columns that meet it.
//
// The work is the rays', not the voxels', so these serve the views with a voxel
// beside or behind the source, which has thousands of candidate pixels for the
// gathers (kernels_gather.hip): 128^3 x 180 views of 256 x 192 on an orbit of 91 mm
// (the volume's corners reach 90.5) Joseph 8.2 ms and Siddon 17.6 against 35.9 and
// 26.1 by the search per voxel and 44 and 41 by the gathers; 80 mm 11.1 and 25.5,
// the search 51 and 32, the gathers 291 and 300.  (They would also be twice as
// fast for few rays before many voxels, one view of 128 x 96 at 256^3 20 us against
// 39, but their FP32 lines put a ray of a source 400 voxels away 4e-5 voxels aside,
// where the gathers' are FP64.)
// Bound: the LDS read-modify-writes of a ray (two words a sample), one after
// another in a lane.  A lane's slots are its own, so nothing is atomic and the
// order of every sum is fixed.
#include <hip/hip_runtime.h>

#include "ray_geometry.hpp"
#include "yk_internal.hpp"

namespace yk {
namespace {

// Column-major ray table of the Joseph scatter: ab1[view][u] = (a1, b1)
// of column u; ab2[view][u][v] = (a2, b2) and pl[view][u][v] = p * L of ray
// (u, v) (0 for a ray the forward projector skips), each column padded to
// nvp = nv + kScatterPad entries with zeros.  Same joseph_ray as the
// forward kernel; the 32 x 32 tile is transposed through LDS so both the
// projection reads and the table writes are contiguous.
__global__ void __launch_bounds__(256)
joseph_scatter_table_kernel(const float* __restrict__ proj, const ProjViewDev* __restrict__ views,
    VolumeGeom g, int nu, int nv, int nvp, float2* __restrict__ ab1, float2* __restrict__ ab2,
    float* __restrict__ pl)
{
    __shared__ float2 s_ab[32][33];
    __shared__ float s_pl[32][33];
    const int i = blockIdx.z;
    const int u0 = blockIdx.x * 32, v0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const ProjViewDev pv = views[i];
    const AxisInfo ax = axis_info(pv.axis, g);
    const float* pi = proj + (size_t)i * nu * nv;
    for (int k = ty; k < 32; k += 8) {
        const int u = u0 + tx, v = v0 + k;
        float2 ab = make_float2(0.f, 0.f);
        float w = 0.f;
        if (u < nu && v < nv) {
            JRay r;
            const bool ok = joseph_ray(pv, ax, u, v, r);
            if (ok) {
                ab = make_float2(r.a2, r.b2);
                w = pi[(size_t)v * nu + u] * r.L;
            }
            if (v == 0) ab1[(size_t)i * nu + u] = ok ? make_float2(r.a1, r.b1) : make_float2(0.f, 0.f);
        }
        s_ab[k][tx] = ab;
        s_pl[k][tx] = w;
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
        const int u = u0 + k, v = v0 + tx;
        if (u < nu && v < nvp) {
            const size_t o = ((size_t)i * nu + u) * nvp + v;
            ab2[o] = s_ab[tx][k];
            pl[o] = s_pl[tx][k];
        }
    }
}

// One lane per (x, y) column of kSepZ voxels, 16 x 16 columns per workgroup.
// Per view the column sits on one main-axis slice s and one first-minor index
// i1, so its candidate rays are whole detector columns u with
// floor(f1(u)) in {i1 - 1, i1}, and in each such column the rays whose f2
// lies in [z0 - 1, z0 + kSepZ).  Those are walked in v order; every ray adds
// p L wa (1 - w2) and p L wa w2 to the two voxels its sample straddles.  The
// sums live in LDS slots private to the lane (slot-major, lane-minor: no
// bank conflicts, no sharing: plain read-modify-write, no atomics), so the
// order of additions per voxel is fixed and the result deterministic.  Candidate ranges come from the FP32
// projective map with 0.05 px of margin; membership is decided only by the
// forward kernel's own f1, f2.
constexpr int kSepZ = 32;
constexpr int kSepU = kScatterPad;  // rays of a column loaded before any is consumed

__global__ void __launch_bounds__(256)
joseph_scatter_kernel(const float2* __restrict__ ab1, const float2* __restrict__ ab2,
    const float* __restrict__ pl, const ProjViewDev* __restrict__ views, const float* __restrict__ c32,
    VolumeGeom g, int nu, int nv, int nvp, int count, int accumulate, float* __restrict__ volume)
{
    __shared__ float slot[(kSepZ + 2) * 256];
    const int lane = threadIdx.x;
    const int x = blockIdx.x * 16 + (lane & 15);
    const int y = blockIdx.y * 16 + (lane >> 4);
    const int z0 = blockIdx.z * kSepZ;
#pragma unroll
    for (int k = 0; k < kSepZ + 2; ++k) slot[k * 256 + lane] = 0.f;
    if (x >= g.nx || y >= g.ny) return;
    const float margin = 0.05f;
    const float zlo = g.oz + float(z0 - 1) * g.vz;
    const float zhi = g.oz + float(z0 + kSepZ) * g.vz;
    const float zmid = g.oz + (float(z0) + 0.5f * float(kSepZ - 1)) * g.vz;
    for (int i = 0; i < count; ++i) {
        const ProjViewDev pv = views[i];
        const AxisInfo ax = axis_info(pv.axis, g);
        const bool xmain = pv.axis == 0;
        const int s = xmain ? x : y, i1 = xmain ? y : x;
        const float c0 = joseph_c0(s, ax.n0);
        const float* c = c32 + (size_t)i * 12;
        const float m0 = (xmain ? g.ox : g.oy) + float(s) * ax.v0;
        const float o1 = xmain ? g.oy : g.ox;
        // detector columns whose rays cross slice s within (i1 - 1, i1 + 1)
        float ua, ub;
        {
            const float ma = o1 + float(i1 - 1) * ax.v1, mb = o1 + float(i1 + 1) * ax.v1;
            const float xa = xmain ? m0 : ma, ya = xmain ? ma : m0;
            const float xb = xmain ? m0 : mb, yb = xmain ? mb : m0;
            const float da = c[8] * xa + c[9] * ya + c[10] * zmid + c[11];
            const float db = c[8] * xb + c[9] * yb + c[10] * zmid + c[11];
            if (!(da > 1e-6f) || !(db > 1e-6f)) continue;
            ua = proj_coord(c, 0, xa, ya, zmid, 1.f / da);
            ub = proj_coord(c, 0, xb, yb, zmid, 1.f / db);
        }
        const int ulo = max(0, int(ceilf(fminf(ua, ub) - margin)));
        const int uhi = min(nu - 1, int(floorf(fmaxf(ua, ub) + margin)));
        for (int u = ulo; u <= uhi; ++u) {
            const float2 q1 = ab1[(size_t)i * nu + u];
            const float f1 = joseph_minor(q1.x, q1.y, c0, ax.n1);
            const float g1 = floorf(f1);
            if (g1 < -1.f || g1 > float(ax.n1 - 1)) continue;
            const int j1 = int(g1);
            const float w1 = f1 - g1;
            float wa;
            if (j1 == i1) wa = 1.f - w1;
            else if (j1 + 1 == i1) wa = w1;
            else continue;
            // rays of column u whose f2 falls in [z0 - 1, z0 + kSepZ)
            const float m1 = o1 + f1 * ax.v1;
            const float xc = xmain ? m0 : m1, yc = xmain ? m1 : m0;
            const float dl = c[8] * xc + c[9] * yc + c[10] * zlo + c[11];
            const float dh = c[8] * xc + c[9] * yc + c[10] * zhi + c[11];
            if (!(dl > 1e-6f) || !(dh > 1e-6f)) continue;
            const float va = proj_coord(c, 4, xc, yc, zlo, 1.f / dl);
            const float vb = proj_coord(c, 4, xc, yc, zhi, 1.f / dh);
            const int vlo = max(0, int(ceilf(fminf(va, vb) - margin)));
            const int vhi = min(nv - 1, int(floorf(fmaxf(va, vb) + margin)));
            // kSepU rays per step, loads first; the column carries kSepU
            // zero-weight pad entries, so a step may run past vhi (rays
            // beyond the candidate range fall outside the slots by f2)
            const float2* q2 = ab2 + ((size_t)i * nu + u) * nvp + vlo;
            const float* w = pl + ((size_t)i * nu + u) * nvp + vlo;
            const int nr = vhi - vlo + 1;
            for (int r0 = 0; r0 < nr; r0 += kSepU) {
                float2 q[kSepU];
                float pw[kSepU];
#pragma unroll
                for (int j = 0; j < kSepU; ++j) {
                    q[j] = q2[r0 + j];
                    pw[j] = w[r0 + j];
                }
#pragma unroll
                for (int j = 0; j < kSepU; ++j) {
                    const float f2 = joseph_minor(q[j].x, q[j].y, c0, ax.n2);
                    const float g2 = floorf(f2);
                    // slot of voxel floor(f2): 0 .. kSepZ covers f2 in
                    // [z0 - 1, z0 + kSepZ); slots of voxels outside the
                    // volume are never stored, which stands in for the
                    // forward kernel's g2 range test
                    const int k = int(g2) - (z0 - 1);
                    const bool live = unsigned(k) <= unsigned(kSepZ);
                    const float w2 = f2 - g2;
                    const float cw = live ? pw[j] * wa : 0.f;
                    float* sk = slot + ((live ? k : 0) * 256 + lane);
                    sk[0] += cw * (1.f - w2);
                    sk[256] += cw * w2;
                }
            }
        }
    }
    const size_t plane = (size_t)g.nx * g.ny;
    const size_t colx = (size_t)y * g.nx + x;
#pragma unroll
    for (int k = 1; k <= kSepZ; ++k) {
        const int z = z0 + k - 1;
        if (z >= g.nz) break;
        const float val = slot[k * 256 + lane];
        float* dst = volume + z * plane + colx;
        *dst = accumulate ? *dst + val : val;
    }
}

// Siddon: the rays of a detector column u share ray_x and ray_y (independent of
// v), hence their XY path: the t-interval of an (x, y) cell and the XY part of the
// volume clip are column constants, and each ray only resolves the z voxels it
// crosses inside that interval.
//
// col_xy[view][u] = (ray_x, ray_y) of column u; ray_wz[view][u][v] =
// (p L, ray_z) of ray (u, v), L = |ray|, each column padded to nvp entries of
// zeros (p L = 0 marks a ray that adds nothing)
__global__ void __launch_bounds__(256)
siddon_scatter_table_kernel(const float* __restrict__ proj, const SiddonViewDev* __restrict__ views,
    int nu, int nv, int nvp, float2* __restrict__ col_xy, float2* __restrict__ ray_wz)
{
    __shared__ float2 s_t[32][33];
    const int i = blockIdx.z;
    const int u0 = blockIdx.x * 32, v0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const SiddonViewDev sv = views[i];
    const float* pi = proj + (size_t)i * nu * nv;
    for (int k = ty; k < 32; k += 8) {
        const int u = u0 + tx, v = v0 + k;
        float2 e = make_float2(0.f, 0.f);
        if (u < nu && v < nv) {
            float src[3], ray[3];
            siddon_ray_geom(sv, u, v, src, ray);
            const float len = sqrtf(ray[0] * ray[0] + ray[1] * ray[1] + ray[2] * ray[2]);
            e = make_float2(pi[(size_t)v * nu + u] * len, ray[2]);
            if (v == 0) col_xy[(size_t)i * nu + u] = make_float2(ray[0], ray[1]);
        }
        s_t[k][tx] = e;
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
        const int u = u0 + k, v = v0 + tx;
        if (u < nu && v < nvp) ray_wz[((size_t)i * nu + u) * nvp + v] = s_t[tx][k];
    }
}

// z-slices per lane column of the Siddon transpose: 16 (18 LDS slots a lane,
// 8 workgroups per CU) measured 18 % faster than 32 at 256^3 x 360; the
// Joseph transpose keeps kSepZ = 32, where 16 measured 12 % slower
constexpr int kSidSepZ = 16;

__global__ void __launch_bounds__(256)
siddon_scatter_kernel(const float2* __restrict__ col_xy, const float2* __restrict__ ray_wz,
    const SiddonViewDev* __restrict__ views, const float* __restrict__ c32, VolumeGeom g, int nu, int nv,
    int nvp, int count, int accumulate, float* __restrict__ volume)
{
    __shared__ float slot[(kSidSepZ + 2) * 256];
    const int lane = threadIdx.x;
    const int x = blockIdx.x * 16 + (lane & 15);
    const int y = blockIdx.y * 16 + (lane >> 4);
    const int z0 = blockIdx.z * kSidSepZ;
#pragma unroll
    for (int k = 0; k < kSidSepZ + 2; ++k) slot[k * 256 + lane] = 0.f;
    if (x >= g.nx || y >= g.ny) return;
    const Box b = volume_box(g);
    const float margin = 0.05f;
    const int zend = min(z0 + kSidSepZ, g.nz);  // one past the block's last slice
    const float xl = b.lo[0] + float(x) * g.vx, xh = b.lo[0] + float(x + 1) * g.vx;
    const float yl = b.lo[1] + float(y) * g.vy, yh = b.lo[1] + float(y + 1) * g.vy;
    const float zl = b.lo[2] + float(z0) * g.vz, zh = b.lo[2] + float(zend) * g.vz;
    const float inv_vz = 1.f / g.vz;
    // only a block holding the volume's first or last slice can see the Z
    // faces of the volume clip bind inside its voxels
    const bool zface = z0 == 0 || zend == g.nz;
    for (int i = 0; i < count; ++i) {
        const float* c = c32 + (size_t)i * 12;
        // detector range of the cell x block (8 corners, FP32 map, margin)
        float umin = 3.0e38f, umax = -3.0e38f, vmin = 3.0e38f, vmax = -3.0e38f;
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float X = (k & 1) ? xh : xl, Y = (k & 2) ? yh : yl, Z = (k & 4) ? zh : zl;
            const float den = c[8] * X + c[9] * Y + c[10] * Z + c[11];
            ok = ok && den > 1e-6f;
            const float rd = 1.f / den;
            const float uu = proj_coord(c, 0, X, Y, Z, rd), vv = proj_coord(c, 4, X, Y, Z, rd);
            umin = fminf(umin, uu); umax = fmaxf(umax, uu);
            vmin = fminf(vmin, vv); vmax = fmaxf(vmax, vv);
        }
        if (!ok) continue;
        const int ulo = max(0, int(ceilf(umin - margin)));
        const int uhi = min(nu - 1, int(floorf(umax + margin)));
        const int vlo = max(0, int(ceilf(vmin - margin)));
        const int vhi = min(nv - 1, int(floorf(vmax + margin)));
        const SiddonViewDev sv = views[i];
        const float sx = sv.src[0], sy = sv.src[1], sz = sv.src[2];
        for (int u = ulo; u <= uhi; ++u) {
            const float2 r = col_xy[(size_t)i * nu + u];
            // XY part of the volume clip and of the cell, shared by the column
            float a0 = 0.f, e0 = 1.f;
            if (!slab_clip(sx, r.x, b.lo[0], b.hi[0], a0, e0)) continue;
            if (!slab_clip(sy, r.y, b.lo[1], b.hi[1], a0, e0)) continue;
            float ca = -3.0e38f, cb = 3.0e38f;
            cell_interval(sx, r.x, b.lo[0], g.vx, x, g.nx, ca, cb);
            cell_interval(sy, r.y, b.lo[1], g.vy, y, g.ny, ca, cb);
            a0 = fmaxf(a0, ca);
            e0 = fminf(e0, cb);
            if (!(e0 > a0)) continue;
            const float2* q = ray_wz + ((size_t)i * nu + u) * nvp + vlo;
            const int nr = vhi - vlo + 1;
            for (int r0 = 0; r0 < nr; r0 += kSepU) {
                float2 e[kSepU];
#pragma unroll
                for (int j = 0; j < kSepU; ++j) e[j] = q[r0 + j];
#pragma unroll
                for (int j = 0; j < kSepU; ++j) {
                    const float pw = e[j].x, rz = e[j].y;
                    float a = a0, t1 = e0;
                    bool live = pw != 0.f;
                    if (zface) live = live && slab_clip(sz, rz, b.lo[2], b.hi[2], a, t1);
                    live = live && t1 > a;
                    if (!live) continue;
                    // Z voxels of the block the ray crosses inside [a, t1]
                    const bool zvalid = fabsf(rz) > 1e-8f;
                    const float rc = zvalid ? 1.f / rz : 0.f;
                    const float za = sz + a * rz, zb = sz + t1 * rz;
                    int ka = int(floorf((fminf(za, zb) - b.lo[2]) * inv_vz));
                    int kb = int(floorf((fmaxf(za, zb) - b.lo[2]) * inv_vz));
                    ka = max(ka, z0);
                    kb = min(kb, zend - 1);
                    for (int k = ka; k <= kb; ++k) {
                        float lo = a, hi = t1;
                        if (zvalid) {
                            const float tl = (b.lo[2] + float(k) * g.vz - sz) * rc;
                            const float th = (b.lo[2] + float(k + 1) * g.vz - sz) * rc;
                            lo = fmaxf(lo, fminf(tl, th));
                            hi = fminf(hi, fmaxf(tl, th));
                        }
                        const float seg = hi - lo;
                        if (seg > 0.f) slot[(k - z0 + 1) * 256 + lane] += pw * seg;
                    }
                }
            }
        }
    }
    const size_t plane = (size_t)g.nx * g.ny;
    const size_t colx = (size_t)y * g.nx + x;
#pragma unroll
    for (int k = 1; k <= kSidSepZ; ++k) {
        const int z = z0 + k - 1;
        if (z >= g.nz) break;
        const float val = slot[k * 256 + lane];
        float* dst = volume + z * plane + colx;
        *dst = accumulate ? *dst + val : val;
    }
}

}  // namespace

void launch_joseph_scatter(const JosephScatterLaunch& p, hipStream_t s)
{
    const int nvp = p.nv + kScatterPad;
    dim3 tb(256), tg((p.nu + 31) / 32, (nvp + 31) / 32, p.count);
    hipLaunchKernelGGL(joseph_scatter_table_kernel, tg, tb, 0, s, p.proj, p.views, p.vol, p.nu, p.nv, nvp, p.ab1,
        p.ab2, p.pl);
    dim3 block(256), grid((p.vol.nx + 15) / 16, (p.vol.ny + 15) / 16, (p.vol.nz + kSepZ - 1) / kSepZ);
    hipLaunchKernelGGL(joseph_scatter_kernel, grid, block, 0, s, p.ab1, p.ab2, p.pl, p.views, p.coeff32,
        p.vol, p.nu, p.nv, nvp, p.count, p.accumulate, p.volume);
    YK_HIP(hipGetLastError());
}

void launch_siddon_scatter(const SiddonScatterLaunch& p, hipStream_t s)
{
    const int nvp = p.nv + kScatterPad;
    dim3 tb(256), tg((p.nu + 31) / 32, (nvp + 31) / 32, p.count);
    hipLaunchKernelGGL(siddon_scatter_table_kernel, tg, tb, 0, s, p.proj, p.views, p.nu, p.nv, nvp, p.col_xy,
        p.ray_wz);
    dim3 block(256), grid((p.vol.nx + 15) / 16, (p.vol.ny + 15) / 16, (p.vol.nz + kSidSepZ - 1) / kSidSepZ);
    hipLaunchKernelGGL(siddon_scatter_kernel, grid, block, 0, s, p.col_xy, p.ray_wz, p.views, p.coeff32,
        p.vol, p.nu, p.nv, nvp, p.count, p.accumulate, p.volume);
    YK_HIP(hipGetLastError());
}

}  // namespace yk
