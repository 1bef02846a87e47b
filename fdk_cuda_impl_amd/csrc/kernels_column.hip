// Transpose of the Joseph projection of untilted views, by detector columns,
// for gfx950.
//
// In such a view all rays (u, v) of a detector column u cross a slice of the
// main axis at one first-minor position f1(u), and at z positions that are
// linear in v.  A wave holds a block of ROWS first-minor rows of one slice,
// lanes along z, and walks the columns that meet it: it gathers a column's rays
// onto the z axis once,
//   h(z) = sum_v p L max(0, 1 - |z - f2(v)|),
// from the four rays (as a rule) next to each voxel, and adds (1 - w) h and w h
// to the two rows beside f1.  A voxel and view thus cost 1.7 columns of four
// candidates of three instructions each, where the gather over both detector
// axes weighs 22 candidates of ten for two voxels.
// The wave's accumulators stay in registers for all views.  X- and Y-main views
// accumulate into volumes of their own, Z-fastest, which a last kernel adds and
// turns to [z][y][x].
// The columns of a slice and block of rows are found by projecting the block's
// ends; their parameters are formed 64 at a time, a column a lane, and handed
// to the wave by lane reads, so a column's candidates differ by lane only in z.
// Bound: the vector memory pipe (16 cycles of a CU for each column and 64 voxels;
// its addressers are 86 % busy, profiles/projectors_counters.txt) and VALU issue (20
// instructions for the same).  Joseph transpose against the gather over both axes: 256^3 x 360 views of 512 x 384
// 15.3 -> 5.8 ms, 128^3 x 120 of 256 x 192 870 -> 426 us, 96^3 x 60 237 -> 169.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ray_geometry.hpp"
#include "yk_internal.hpp"

namespace yk {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
constexpr int kRsrcWord3 = 0x00020000;  // raw buffer, 32-bit data format

__device__ __forceinline__ floatx4 load4(__amdgpu_buffer_rsrc_t r, int offset)
{
    return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, offset, 0, 0));
}

__device__ __forceinline__ float lane_value(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

__global__ void column_clear_kernel(int* __restrict__ flag) { *flag = 0; }

// p L of every ray, [view][u][kColumnPad + v], with kColumnPad zeros on either
// side of a column; a value that is not finite raises *flag, and the candidates
// that do not meet a voxel are then skipped rather than weighed with zero
__global__ void __launch_bounds__(256)
joseph_column_table_kernel(const float* __restrict__ proj, const ProjViewDev* __restrict__ views, VolumeGeom g, int nu, int nv,
    int pitch, float* __restrict__ q, int* __restrict__ flag)
{
    __shared__ float tile[32][33];
    const int u0 = blockIdx.x * 32, e0 = blockIdx.y * 32, i = blockIdx.z;
    const ProjViewDev pv = views[i];
    const AxisInfo ax = axis_info(pv.axis, g);
    bool bad = false;
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int u = u0 + int(threadIdx.x), v = e0 + k - kColumnPad;
        float w = 0.f;
        if (u < nu && v >= 0 && v < nv) {
            JRay r;
            if (joseph_ray(pv, ax, u, v, r)) w = proj[((size_t)i * nv + v) * nu + u] * r.L;
            bad = bad || !(fabsf(w) <= 3.4e38f);
        }
        tile[k][threadIdx.x] = w;
    }
    if (bad) atomicOr(flag, 1);
    __syncthreads();
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int u = u0 + k, e = e0 + int(threadIdx.x);
        if (u < nu && e < pitch) q[((size_t)i * nu + u) * pitch + e] = tile[threadIdx.x][k];
    }
}

template <int ROWS, int KZ, bool SAFE>
__device__ __forceinline__ void column_gather(const float* __restrict__ q, const GatherViewDev* __restrict__ gviews, int axis, const AxisInfo& ax, int nu, int nv, int pitch, int count, int s, int j0,
    int z0, float (&acc)[ROWS][KZ])
{
    const int lane = int(threadIdx.x & 63);
    const double c0 = double(joseph_c0(s, ax.n0)), h1 = 0.5 * double(ax.n1 - 1);
    const float vmid = 0.5f * float(nv - 1), vpad = vmid + float(kColumnPad);
    // the block's end rows, as voxel indices (the volume's ends bound them)
    const float row_a = float(j0 - 1), row_b = float(min(j0 + ROWS, ax.n1));
    float zc[KZ];
#pragma unroll
    for (int k = 0; k < KZ; ++k) zc[k] = float(z0 + lane + 64 * k) - 0.5f * float(ax.n2 - 1);
#pragma unroll 1
    for (int i = 0; i < count; ++i) {
        const GatherViewDev& m = gviews[i];
        if (m.axis != axis) continue;
        const bool xmain = axis == 0;
        // columns that can lie within a row of the block: 0.05 pixels of margin
        // for the FP32 map
        const float ms = xmain ? m.mu[0] : m.mu[1], mr = xmain ? m.mu[1] : m.mu[0];
        const float ds = xmain ? m.md[0] : m.md[1], dr = xmain ? m.md[1] : m.md[0];
        const float us = fmaf(ms, float(s), m.mu[3]), des = fmaf(ds, float(s), m.md[3]);
        const float ua = fmaf(mr, row_a, us) / fmaf(dr, row_a, des), ub = fmaf(mr, row_b, us) / fmaf(dr, row_b, des);
        const int lo = __builtin_amdgcn_readfirstlane(int(fmaxf(0.f, ceilf(fminf(ua, ub) - 0.05f))));
        const int hi = __builtin_amdgcn_readfirstlane(int(fminf(float(nu - 1), floorf(fmaxf(ua, ub) + 0.05f))));
        const float* const qi = q + (size_t)i * nu * pitch;
#pragma unroll 1
        for (int first = lo; first <= hi; first += 64) {
            const int u = first + lane;
            // (FP64: the terms of a position are a thousand times the weights)
            const double d0 = fma(double(u), m.d[1], m.d[0]);
            const double tau = (c0 - m.src[0]) / d0;
            const double f1 = fma(fma(double(u), m.e1[1], m.e1[0]), tau, m.src[1]) + h1;
            const double floor1 = floor(f1);
            // (a row outside the block where the lane has no column)
            const int row = u <= hi && d0 != 0.0 ? int(fmin(fmax(floor1, -2.0), 1e6)) - j0 : -2;
            const float t_w = float(f1 - floor1), t_slope = float(tau * m.e2[2]), t_inv = 1.f / t_slope;
            const float t_q = float(fma(fma(double(vmid), m.e2[2], fma(double(u), m.e2[1], m.e2[0])), tau, m.src[2]));
            // first candidate of z: ceil(vmid + (z - q) / slope - 1 / |slope|), 0.01 pixels early
            const float t_v = vpad - fabsf(t_inv) - 0.01f;
            const unsigned long long more = __ballot(fabsf(t_inv) > 1.98f);  // more than four candidates
#pragma unroll
            for (int r = -1; r < ROWS; ++r) {
                unsigned long long mask = __ballot(row == r);
                while (mask) {
                    const int l = __builtin_ctzll(mask);
                    mask &= mask - 1;
                    const float w = lane_value(t_w, l), qz = lane_value(t_q, l), slope = lane_value(t_slope, l);
                    const float inv = lane_value(t_inv, l), v_off = lane_value(t_v, l);
                    // a start before the column's first pad or in its last three
                    // floats, which are pads, reads zeros (out of the buffer's range)
                    const __amdgpu_buffer_rsrc_t col = __builtin_amdgcn_make_buffer_rsrc(
                        const_cast<float*>(qi + (size_t)(first + l) * pitch), 0, (pitch - 3) * 4, kRsrcWord3);
                    floatx4 p[KZ];
                    float d[KZ], h[KZ];
                    int off[KZ];
#pragma unroll
                    for (int k = 0; k < KZ; ++k) {
                        const float t = zc[k] - qz;
                        const float v = ceilf(fmaf(t, inv, v_off));  // + kColumnPad
                        d[k] = fmaf(-slope, v - vpad, t);
                        off[k] = int(v) * 4;
                        p[k] = load4(col, off[k]);
                    }
                    auto weigh = [&](int k, float x, float sum) {
                        const float a = __builtin_amdgcn_fmed3f(1.f - fabsf(d[k]), 0.f, 1.f);
                        d[k] -= slope;
                        return !SAFE || a > 0.f ? fmaf(a, x, sum) : sum;
                    };
#pragma unroll
                    for (int k = 0; k < KZ; ++k) {
                        h[k] = weigh(k, p[k].x, 0.f);
                        h[k] = weigh(k, p[k].y, h[k]);
                        h[k] = weigh(k, p[k].z, h[k]);
                        h[k] = weigh(k, p[k].w, h[k]);
                    }
                    if ((more >> l) & 1) {
#pragma unroll
                        for (int k = 0; k < KZ; ++k) p[k] = load4(col, off[k] + 16);
#pragma unroll
                        for (int k = 0; k < KZ; ++k) {
                            h[k] = weigh(k, p[k].x, h[k]);
                            h[k] = weigh(k, p[k].y, h[k]);
                            h[k] = weigh(k, p[k].z, h[k]);
                            h[k] = weigh(k, p[k].w, h[k]);
                        }
                    }
#pragma unroll
                    for (int k = 0; k < KZ; ++k) {
                        if (r >= 0) acc[r < 0 ? 0 : r][k] = fmaf(1.f - w, h[k], acc[r < 0 ? 0 : r][k]);
                        if (r + 1 < ROWS && (!SAFE || w > 0.f)) {
                            const int n = r + 1 < ROWS ? r + 1 : 0;
                            acc[n][k] = fmaf(w, h[k], acc[n][k]);
                        }
                    }
                }
            }
        }
    }
}

// volumes [slice][row][z] of the X- (part_x) and Y-main views; blockIdx.z runs
// over the z blocks of either axis that has views
template <int ROWS, int KZ>
__global__ void __launch_bounds__(64 * kColumnSlices, 4)
joseph_column_transpose_kernel(const float* __restrict__ q, float* __restrict__ part_x, float* __restrict__ part_y,
    const GatherViewDev* __restrict__ gviews, const int* __restrict__ flag, VolumeGeom g, int nu, int nv, int pitch, int count)
{
    const bool both = part_x && part_y;
    const int axis = both ? int(blockIdx.z & 1u) : (part_x ? 0 : 1);
    const int z0 = (both ? int(blockIdx.z >> 1) : int(blockIdx.z)) * 64 * KZ;
    const AxisInfo ax = axis_info(axis, g);
    const int s = __builtin_amdgcn_readfirstlane(int(blockIdx.x) * kColumnSlices + int(threadIdx.x >> 6));
    const int j0 = int(blockIdx.y) * ROWS;
    if (s >= ax.n0 || j0 >= ax.n1) return;  // whole wave
    float acc[ROWS][KZ];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int k = 0; k < KZ; ++k) acc[r][k] = 0.f;
    if (__builtin_amdgcn_readfirstlane(*flag) == 0)
        column_gather<ROWS, KZ, false>(q, gviews, axis, ax, nu, nv, pitch, count, s, j0, z0, acc);
    else
        column_gather<ROWS, KZ, true>(q, gviews, axis, ax, nu, nv, pitch, count, s, j0, z0, acc);
    float* const out = axis == 0 ? part_x : part_y;
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int k = 0; k < KZ; ++k) {
            const int z = z0 + int(threadIdx.x & 63) + 64 * k;
            if (j0 + r < ax.n1 && z < ax.n2) out[((size_t)s * ax.n1 + (j0 + r)) * ax.n2 + z] = acc[r][k];
        }
}

// volume (+)= part_x [x][y][z] + part_y [y][x][z], either of which may be null
__global__ void __launch_bounds__(256)
joseph_column_sum_kernel(const float* __restrict__ part_x, const float* __restrict__ part_y, float* __restrict__ volume, int nx,
    int ny, int nz, int accumulate)
{
    __shared__ float tile[32][33];
    const int z0 = blockIdx.x * 32, x0 = blockIdx.y * 32, y = blockIdx.z;
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int x = x0 + k, z = z0 + int(threadIdx.x);
        float v = 0.f;
        if (x < nx && z < nz) {
            if (part_x) v = part_x[((size_t)x * ny + y) * nz + z];
            if (part_y) v += part_y[((size_t)y * nx + x) * nz + z];
        }
        tile[k][threadIdx.x] = v;
    }
    __syncthreads();
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int z = z0 + k, x = x0 + int(threadIdx.x);
        if (x >= nx || z >= nz) continue;
        float* dst = volume + ((size_t)z * ny + y) * nx + x;
        *dst = accumulate ? *dst + tile[threadIdx.x][k] : tile[threadIdx.x][k];
    }
}

template <int ROWS, int KZ>
void launch_blocks(const ColumnTransposeLaunch& p, hipStream_t s)
{
    const VolumeGeom& g = p.vol;
    const int n0 = std::max(p.part_x ? g.nx : 0, p.part_y ? g.ny : 0), n1 = std::max(p.part_x ? g.ny : 0, p.part_y ? g.nx : 0);
    dim3 grid((n0 + kColumnSlices - 1) / kColumnSlices, (n1 + ROWS - 1) / ROWS,
        (g.nz + 64 * KZ - 1) / (64 * KZ) * (p.part_x && p.part_y ? 2 : 1));
    hipLaunchKernelGGL((joseph_column_transpose_kernel<ROWS, KZ>), grid, dim3(64 * kColumnSlices), 0, s, p.q, p.part_x, p.part_y,
        p.gviews, p.flag, g, p.nu, p.nv, p.pitch, p.count);
}

// Rows a wave: a block of ROWS walks the columns of ROWS + 1, so the more rows
// the better, as long as they leave waves for the GPU's 1024 SIMDs (four are
// resident on each).  With 16, 8 and 4 rows: 256^3 x 360 views (8192 waves of
// 16 rows) 5.84, 6.23 and 7.01 ms, 200^3 x 100 (5200) 1.23, 1.11 and 1.20 ms;
// 128^3 x 120 (4096 waves of 8 rows) 540, 426 and 458 us, 96^3 x 60 (2304) 280,
// 198 and 169 us.
template <int KZ>
void launch_rows(const ColumnTransposeLaunch& p, hipStream_t s)
{
    const VolumeGeom& g = p.vol;
    auto waves = [&](int rows) {
        const long blocks = (p.part_x ? long(g.nx) * ((g.ny + rows - 1) / rows) : 0) +
            (p.part_y ? long(g.ny) * ((g.nx + rows - 1) / rows) : 0);
        return blocks * ((g.nz + 64 * KZ - 1) / (64 * KZ));
    };
    if (waves(16) >= 8192) launch_blocks<16, KZ>(p, s);
    else if (waves(8) >= 4096) launch_blocks<8, KZ>(p, s);
    else launch_blocks<4, KZ>(p, s);
}

}  // namespace

void launch_joseph_column_transpose(const ColumnTransposeLaunch& p, hipStream_t s)
{
    const VolumeGeom& g = p.vol;
    hipLaunchKernelGGL(column_clear_kernel, dim3(1), dim3(1), 0, s, p.flag);
    dim3 tg((p.nu + 31) / 32, (p.pitch + 31) / 32, p.count);
    hipLaunchKernelGGL(joseph_column_table_kernel, tg, dim3(32, 8), 0, s, p.proj, p.views, g, p.nu, p.nv, p.pitch, p.q, p.flag);
    // z blocks of 64 to 256 voxels, as even as they come
    const int groups = (g.nz + 63) / 64, blocks = (groups + kColumnGroups - 1) / kColumnGroups;
    switch ((groups + blocks - 1) / blocks) {
    case 1: launch_rows<1>(p, s); break;
    case 2: launch_rows<2>(p, s); break;
    case 3: launch_rows<3>(p, s); break;
    default: launch_rows<4>(p, s); break;
    }
    dim3 sg((g.nz + 31) / 32, (g.nx + 31) / 32, g.ny);
    hipLaunchKernelGGL(joseph_column_sum_kernel, sg, dim3(32, 8), 0, s, p.part_x, p.part_y, p.volume, g.nx, g.ny, g.nz,
        p.accumulate);
    YK_HIP(hipGetLastError());
}

}  // namespace yk
