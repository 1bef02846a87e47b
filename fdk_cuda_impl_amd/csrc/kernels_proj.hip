// Flat-panel forward projectors and their exact transposes for gfx950.
//
// Joseph: per ray, sum over every slice of the per-view main axis of the
// bilinear (minor-axis) sample of the volume at the ray's crossing, times
// sqrt(v0^2 + (a1 v1)^2 + (a2 v2)^2) (fp_joseph_kernel,
// src/FlatFpBp/FP/kernels/YkFPKernels.cu:10-202; axis conventions
// src/common/cuda/operators/YkOperatorKernelTypes.cuh:133-275).  The volume is
// read with software bilinear in place of a 3-D texture; for X-main-axis
// views a [z][x][y] copy keeps the minor-axis gathers contiguous.
//
// Siddon: exact voxel walk from the source to the pixel centre clipped to
// t in [0, 1] and the volume box (siddon_fp_kernel,
// src/FlatFpBp/FP/kernels/YkFPSiddonKernel.cu:19-124); voxel boundaries are
// recomputed from integer indices instead of accumulated.
//
// Transposes are deterministic (no atomics).  The gathers here serve the views that
// kernels_gather.hip, kernels_column.hip and kernels_scatter.hip leave: for each voxel and
// view the candidate rays are the detector pixels inside the projection of the
// voxel's support, and each is re-evaluated with exactly the arithmetic of the
// forward kernel (shared functions below, FP contraction off).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ray_geometry.hpp"
#include "yk_internal.hpp"

namespace yk {
namespace {

// minor-axis sample position of slice s
__device__ __forceinline__ void joseph_sample(const JRay& r, const AxisInfo& ax, int s, float& f1, float& f2)
{
    const float c0 = joseph_c0(s, ax.n0);
    f1 = joseph_minor(r.a1, r.b1, c0, ax.n1);
    f2 = joseph_minor(r.a2, r.b2, c0, ax.n2);
}

// slices whose sample can touch the volume: -1 < f < n on both minor axes
__device__ __forceinline__ void joseph_slice_range(const JRay& r, const AxisInfo& ax, int& lo, int& hi)
{
    float slo = 0.f, shi = float(ax.n0 - 1);
    const float h0 = 0.5f * float(ax.n0 - 1);
    const float a[2] = { r.a1, r.a2 };
    const float b[2] = { r.b1 + 0.5f * float(ax.n1 - 1), r.b2 + 0.5f * float(ax.n2 - 1) };
    const float n[2] = { float(ax.n1), float(ax.n2) };
    for (int k = 0; k < 2; ++k) {
        if (fabsf(a[k]) > 1e-12f) {
            float t0 = (-1.f - b[k]) / a[k] + h0;
            float t1 = (n[k] - b[k]) / a[k] + h0;
            if (t0 > t1) { const float t = t0; t0 = t1; t1 = t; }
            slo = fmaxf(slo, t0);
            shi = fminf(shi, t1);
        } else if (b[k] <= -1.f || b[k] >= n[k]) {
            lo = 1; hi = 0;
            return;
        }
    }
    // one slice of margin on each side; out-of-range samples weigh zero anyway
    lo = max(0, int(floorf(slo)) - 1);
    hi = min(ax.n0 - 1, int(ceilf(shi)) + 1);
}

// One ray per lane, 64 x 4 rays per workgroup.  The lanes of a wave march
// the same slice index (the union of their slice ranges, lanes outside their
// own range weigh zero), so a sample costs four unconditional loads at
// clamped in-volume positions, with the off-volume taps zeroed in the weights;
// four samples are issued before any is consumed.
__global__ void __launch_bounds__(256)
joseph_fp_kernel(const float* __restrict__ vol, const float* __restrict__ vol_t,
    float* __restrict__ proj, const ProjViewDev* __restrict__ views, VolumeGeom g,
    int nu, int nv, int accumulate)
{
    const int u = blockIdx.x * 64 + threadIdx.x;
    const int v = blockIdx.y * 4 + threadIdx.y;
    const int i = blockIdx.z;
    const bool pix = u < nu && v < nv;
    const ProjViewDev pv = views[i];
    const AxisInfo ax = axis_info(pv.axis, g);
    // memory strides of (s, i1, i2)
    const float* base;
    size_t st0, st2;
    if (pv.axis == 0) { base = vol_t; st0 = (size_t)g.ny; st2 = (size_t)g.nx * g.ny; }
    else if (pv.axis == 1) { base = vol; st0 = (size_t)g.nx; st2 = (size_t)g.nx * g.ny; }
    else { base = vol; st0 = (size_t)g.nx * g.ny; st2 = (size_t)g.nx; }
    JRay r{};
    int lo = 1, hi = 0;
    if (pix && joseph_ray(pv, ax, u, v, r)) joseph_slice_range(r, ax, lo, hi);
    // wave-wide slice range
    int wlo = lo <= hi ? lo : 0x7fffffff, whi = lo <= hi ? hi : -1;
    for (int off = 32; off > 0; off >>= 1) {
        wlo = min(wlo, __shfl_xor(wlo, off, 64));
        whi = max(whi, __shfl_xor(whi, off, 64));
    }
    const int n1 = ax.n1, n2 = ax.n2;
    float acc = 0.f;
    constexpr int kUnroll = 4;
    for (int s0 = wlo; s0 <= whi; s0 += kUnroll) {
        float t[kUnroll][4], wa[kUnroll], wb[kUnroll], wc[kUnroll], wd[kUnroll];
#pragma unroll
        for (int k = 0; k < kUnroll; ++k) {
            const int s = min(s0 + k, whi);
            float f1, f2;
            joseph_sample(r, ax, s, f1, f2);
            const float g1 = floorf(f1), g2 = floorf(f2);
            const float w1 = f1 - g1, w2 = f2 - g2;
            const bool live = s0 + k <= whi && s >= lo && s <= hi && g1 >= -1.f && g2 >= -1.f &&
                g1 <= float(n1 - 1) && g2 <= float(n2 - 1);
            const int j1 = live ? int(g1) : 0, j2 = live ? int(g2) : 0;
            // taps (j1 + a, j2 + b) inside the volume, the others weigh zero
            const bool a0 = j1 >= 0, a1 = j1 + 1 < n1, b0 = j2 >= 0, b1 = j2 + 1 < n2;
            const float x0 = live && a0 ? 1.f - w1 : 0.f, x1 = live && a1 ? w1 : 0.f;
            const float y0 = b0 ? 1.f - w2 : 0.f, y1 = b1 ? w2 : 0.f;
            wa[k] = x0 * y0; wb[k] = x1 * y0; wc[k] = x0 * y1; wd[k] = x1 * y1;
            const int c1 = max(j1, 0), c1b = min(j1 + 1, n1 - 1);
            const int c2 = max(j2, 0), c2b = min(j2 + 1, n2 - 1);
            const float* sl = base + (size_t)s * st0;
            t[k][0] = sl[(size_t)c2 * st2 + c1];
            t[k][1] = sl[(size_t)c2 * st2 + c1b];
            t[k][2] = sl[(size_t)c2b * st2 + c1];
            t[k][3] = sl[(size_t)c2b * st2 + c1b];
        }
#pragma unroll
        for (int k = 0; k < kUnroll; ++k)
            acc += (wa[k] * t[k][0] + wb[k] * t[k][1]) + (wc[k] * t[k][2] + wd[k] * t[k][3]);
    }
    if (!pix) return;
    const float out = lo <= hi ? acc * r.L : 0.f;
    float* dst = proj + ((size_t)i * nv + v) * nu + u;
    *dst = accumulate ? *dst + out : out;
}

// store of a projected ray's value, or of the algebraic solvers' weighted
// residual with it, in place of a pass of its own (SART at 64 x 60 x 48 x 40
// views 0.79 -> 0.68 ms)
__device__ __forceinline__ void store_ray(float* proj, int i, int nu, int nv, int u, int v, float out, const FpStore& st)
{
    const size_t in_view = (size_t)v * nu + u, at = (size_t)i * nv * nu + in_view;
    if (st.mode == FpStore::kSet) {
        proj[at] = out;
    } else if (st.mode == FpStore::kAdd) {
        proj[at] += out;
    } else {
        const float r = st.b[(size_t)i * st.b_view + in_view] - out, w = st.row[at];
        proj[at] = st.mode == FpStore::kResidualDivide ? (w > st.eps ? r / w : 0.f) : r * w;
    }
}

// final store of one Joseph ray: the sum times the ray's step length, or
// zero for a ray that misses the volume
__device__ __forceinline__ void finish_joseph(float* proj, int i, int nu, int nv, int u, int v, bool pix,
    bool hit, float acc, float L, const FpStore& st)
{
    if (!pix) return;
    store_ray(proj, i, nu, nv, u, v, hit ? acc * L : 0.f, st);
}

// Paired guarded volume copies of the slab projections.  A guarded copy
// has kJosephGuard zero planes on both sides of both minor axes; its paired
// form stores, at entry (slice c, row r, column e), the two guarded values
// of rows r and r + 1 in column e.  One 16-byte load at (c, r, e) then
// returns the four taps (r, e), (r + 1, e), (r, e + 1), (r + 1, e + 1) of a
// bilinear sample: a wave64 load of 8 or 16 bytes per lane takes 16 cycles
// of a CU's vector memory pipe on gfx950, so the one wider load halves the
// cost of two 8-byte row loads.  Rows run 0 .. n_r + 2 guards - 2 (the last
// row pairs with the trailing guard plane).
constexpr int kJosephGuard = 2;
typedef float float4u __attribute__((ext_vector_type(4), aligned(8)));

// Joseph projection for separable views (main axis X or Y, detV along Z
// only).  A wave takes one detector column u and 64 K of its rays in v.  a1,
// b1 - hence f1, its weight and its two tap rows in a slice - are the same for
// all of them, so per slice the wave interpolates the tap rows once, lanes
// along z (two coalesced 16-byte loads of a Z-fastest copy a lane), leaves the
// column in LDS, and each ray takes a linear sample of it, lanes along v.  A
// sample is two LDS words and a few FP32 instructions where a bilinear gather
// of 16 bytes took 16 cycles of the CU's vector memory pipe; the loads of the
// next slice are in flight while a slice is sampled.
// The copy has kJosephGuard zero planes on both sides of both minor axes, and
// sample positions are clamped to [-2, n], so a position outside (-1, n) reads
// only zeros and no sample is tested for range.
// Bound: the chain of a slice (load, interpolation, LDS, samples), with the vector
// memory pipe 64 %, the LDS 50 % and the VALU up to 97 % busy
// (profiles/projectors_counters.txt; without the volume's loads 25 % less time,
// without loads and LDS reads 47 %).  Six waves a SIMD hide the chain: with four 4 %
// slower, with eight the spills cost as much again.  Copies included, with gathers
// -> here: 256^3 x 360 views of 512 x 384 9.2 -> 5.7 ms, 512^3 x 90 of 1024 x 768 23.7
// -> 15.7 ms, 128^3 x 12 of 256 x 192 69 -> 55 us.
constexpr int kColumnChunk = 256;  // z a wave loads at a time, four a lane
// values of a copy's row: whole 16-byte groups
__host__ __device__ __forceinline__ int column_pitch(int nz) { return (nz + 2 * kJosephGuard + 3) & ~3; }

constexpr int kColumnWaves = 8;
// A column's slices are summed in this many equal parts, then the parts in
// order, however many waves take them: a ray has the same bits in every call
// (256^3 x 360 views 5.70 -> 5.78 ms for the parts' sums).
constexpr int kColumnParts = 8;

template <int K, bool SPLIT>
__global__ void __launch_bounds__(64 * kColumnWaves, 6)
joseph_fp_column_kernel(const float* __restrict__ vzx, const float* __restrict__ vzy,
    float* __restrict__ proj, const ProjViewDev* __restrict__ views, VolumeGeom g,
    int nu, int nv, int count, FpStore st)
{
    // per wave, 64 slices at a time: x = weight of the second tap row, y =
    // byte offset of the first row at the column's first z, z, w = tau and
    // base of f = base + tau e, a ray's position from there (e: its z offset
    // from the detector's middle row, the same in every slice); and the
    // largest f, two less than the column's values
    __shared__ float4 tab[kColumnWaves][64];
    __shared__ float tab_top[kColumnWaves][64];
    extern __shared__ float4 column_raw[];
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = int(threadIdx.x & 63);
    // The waves of a workgroup take one column of consecutive views (their
    // rays nearly coincide, so the repeats of a tap row hit the CU's L1) or,
    // SPLIT, equal numbers of the parts of one column of one view, added at the
    // end: for calls of too few columns to fill the GPU.
    // Columns are remapped so that each XCD (workgroups go round-robin to the
    // 8 XCDs; gridDim.x is a multiple of 8) sweeps a contiguous range of them,
    // whose neighbouring rays share tap rows in its L2.
    const int u = int(blockIdx.x & 7u) * int(gridDim.x >> 3) + int(blockIdx.x >> 3);
    const int v0 = int(blockIdx.y) * 64 * K;
    const int waves = int(blockDim.x >> 6);
    const int i = SPLIT ? int(blockIdx.z) : int(blockIdx.z) * waves + wave;
    if (u >= nu || i >= count) return;  // whole wave, SPLIT: whole workgroup
    const int words = column_pitch(g.nz);
    float* const column = reinterpret_cast<float*>(column_raw) + wave * words;
    // SPLIT: the parts' sums, 64 K floats each, behind the columns
    float* const sums = reinterpret_cast<float*>(column_raw) + waves * words;
    const ProjViewDev pv = views[i];
    const AxisInfo ax = axis_info(pv.axis, g);
    const float s0 = pick(ax.p0, pv.src[0], pv.src[1], 0.f), s1 = pick(ax.p1, pv.src[0], pv.src[1], 0.f), s2 = pv.src[2];
    const float dv2 = pv.detV[2], vmid = 0.5f * float(nv - 1);
    const float h1 = 0.5f * float(ax.n1 - 1), h2 = 0.5f * float(ax.n2 - 1) + float(kJosephGuard);
    // the column's offsets from the source (at the middle row)
    const float d0 = (pick(ax.p0, pv.detS[0], pv.detS[1], 0.f) + float(u) * pick(ax.p0, pv.detU[0], pv.detU[1], 0.f)) - s0;
    const float d1 = (pick(ax.p1, pv.detS[0], pv.detS[1], 0.f) + float(u) * pick(ax.p1, pv.detU[0], pv.detU[1], 0.f)) - s1;
    const float d2 = (pv.detS[2] + float(u) * pv.detU[2] + vmid * dv2) - s2;
    const float rd0 = d0 != 0.f ? 1.f / d0 : 0.f;
    float e[K], acc[K], total[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        // rays past the last one repeat it and store nothing
        e[k] = (float(min(v0 + 64 * k + lane, nv - 1)) - vmid) * dv2;
        acc[k] = total[k] = 0.f;
    }
    const float eF = (float(v0) - vmid) * dv2, eE = (float(min(v0 + 64 * K, nv) - 1) - vmid) * dv2;
    // slices in which the column can lie inside (-1, n) on the first minor
    // axis, with a slice of margin (z needs no range: outside reads zeros)
    int wlo = 1, whi = 0;
    if (d0 != 0.f) {
        JRay r{};
        r.a1 = d1 * rd0;
        r.b1 = s1 - r.a1 * s0;
        joseph_slice_range(r, ax, wlo, whi);
    }
    wlo = __builtin_amdgcn_readfirstlane(wlo);
    whi = __builtin_amdgcn_readfirstlane(whi);
    const int part = (whi - wlo + kColumnParts) / kColumnParts;  // slices
    int part_at = 0, part_top = kColumnParts;
    if constexpr (SPLIT) {
        const int parts = kColumnParts / waves;
        part_at = wave * parts;
        part_top = part_at + parts;
        wlo += part_at * part;
        whi = min(whi, wlo + parts * part - 1);
    }
    int part_end = wlo + part - 1;
    auto end_part = [&]() {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if constexpr (SPLIT) sums[(part_at * K + k) * 64 + lane] = acc[k];
            else total[k] += acc[k];
            acc[k] = 0.f;
        }
        ++part_at;
        part_end += part;
    };
    const int p2 = column_pitch(ax.n2);
    const size_t slice_bytes = size_t(ax.n1 + 2 * kJosephGuard) * p2 * 4u;
    const float f1max = float(ax.n1), f2max = float(ax.n2 + kJosephGuard);
    float4* const t = tab[wave];
    float* const tt = tab_top[wave];
    const char* sl = reinterpret_cast<const char*>(pv.axis == 0 ? vzx : vzy) + size_t(wlo) * slice_bytes;
    float4 ra, rb;
    // Issues the loads of a column of the slice at p (rows at byte offset o,
    // which is a multiple of 16, top + 2 values): four values of either tap
    // row a lane.
    const float first = float(4 * lane - 2);
    auto load = [&](const char* p, unsigned o, float top) {
        if (first < top) {
            const char* a = p + (o + unsigned(lane) * 16u);
            ra = *reinterpret_cast<const float4*>(a);
            rb = *reinterpret_cast<const float4*>(a + size_t(p2) * 4u);
        }
    };
    auto lerp4 = [](float w, const float4& a, const float4& b) {
        return make_float4(fmaf(w, b.x - a.x, a.x), fmaf(w, b.y - a.y, a.y), fmaf(w, b.z - a.z, a.z), fmaf(w, b.w - a.w, a.w));
    };
    for (int c = wlo; c <= whi; c += 64) {
        const int end = min(c + 63, whi);
        int chunks;
        {
            // the column's line in this slice: f = s + d (c0 - s0) / d0
            const float c0 = joseph_c0(min(c + lane, end), ax.n0);
            const float tau = (c0 - s0) * rd0;
            const float f1 = __builtin_amdgcn_fmed3f(fmaf(d1, tau, s1) + h1, -2.f, f1max);
            const float q = fmaf(d2, tau, s2);
            const float fF = __builtin_amdgcn_fmed3f(fmaf(eF, tau, q + h2), 0.f, f2max);
            const float fE = __builtin_amdgcn_fmed3f(fmaf(eE, tau, q + h2), 0.f, f2max);
            // the rays' positions are monotonic in v up to rounding: one z to
            // spare below the lower end, and above the upper end's second tap
            // (from a whole 16-byte group on)
            const int zlo = max(int(fminf(fF, fE)) - 1, 0) & ~3, zhi = min(int(fmaxf(fF, fE)) + 2, ax.n2 + 2 * kJosephGuard - 1);
            const int row = int(floorf(f1)) + kJosephGuard;
            t[lane] = make_float4(__builtin_amdgcn_fractf(f1), __uint_as_float(unsigned(row * p2 + zlo) * 4u), tau,
                q + (h2 - float(zlo)));
            tt[lane] = float(zhi - zlo - 1);
            chunks = (zhi - zlo + kColumnChunk) / kColumnChunk;
            for (int off = 32; off > 0; off >>= 1) chunks = max(chunks, __shfl_xor(chunks, off, 64));
            chunks = __builtin_amdgcn_readfirstlane(chunks);
        }
        __builtin_amdgcn_wave_barrier();
        // cur is sampled while nxt loads, and the entry after it is read
        float4 cur = t[0], nxt = t[min(1, end - c)];
        float ctop = tt[0], ntop = tt[min(1, end - c)];
        load(sl, __float_as_uint(cur.y), ctop);
        for (int s = c; s <= end;) {
            for (const int stop = min(end, part_end); s <= stop; ++s) {
                const float4 after = t[min(s + 2, end) - c];
                const float atop = tt[min(s + 2, end) - c];
                float4* const col4 = reinterpret_cast<float4*>(column);
                if (first < ctop) col4[lane] = lerp4(cur.x, ra, rb);
                if (chunks > 1) {  // a longer column: the rest, not loaded ahead
                    const char* p = sl + __float_as_uint(cur.y);
                    for (int z = kColumnChunk + 4 * lane; z < int(ctop) + 2; z += kColumnChunk)
                        col4[z / 4] = lerp4(cur.x, *reinterpret_cast<const float4*>(p + size_t(z) * 4u),
                                            *reinterpret_cast<const float4*>(p + (size_t(z) + p2) * 4u));
                }
                if (s < whi) {
                    // (past the table's last slice: reloads it, unused)
                    load(sl + (s < end ? slice_bytes : 0), __float_as_uint(nxt.y), ntop);
                    sl += slice_bytes;
                }
                __builtin_amdgcn_wave_barrier();
                float lo[K], hi[K], w[K];
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const float f = __builtin_amdgcn_fmed3f(fmaf(e[k], cur.z, cur.w), 0.f, ctop);
                    const float* p = column + int(f);
                    lo[k] = p[0];
                    hi[k] = p[1];
                    w[k] = __builtin_amdgcn_fractf(f);
                }
#pragma unroll
                for (int k = 0; k < K; ++k) acc[k] += fmaf(w[k], hi[k] - lo[k], lo[k]);
                __builtin_amdgcn_wave_barrier();
                cur = nxt;
                ctop = ntop;
                nxt = after;
                ntop = atop;
            }
            if (s > part_end) end_part();
        }
    }
    auto store = [&](int v, float sum) {
        if (v >= nv) return;
        JRay r{};
        store_ray(proj, i, nu, nv, u, v, joseph_ray(pv, ax, u, v, r) ? sum * r.L : 0.f, st);
    };
    if constexpr (SPLIT) {
        while (part_at < part_top) end_part();  // the last one, and any that no slice is left for
        __syncthreads();
        for (int k = wave; k < K; k += waves) {
            float sum = 0.f;
            for (int p = 0; p < kColumnParts; ++p) sum += sums[(p * K + k) * 64 + lane];
            store(v0 + 64 * k + lane, sum);
        }
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) store(v0 + 64 * k + lane, total[k] + acc[k]);
    }
}

// Joseph projection for any X- or Y-main view set (tilted detectors, lifted
// sources), one lane per ray as joseph_fp_kernel, over paired slab copies:
// rows along z and columns along the first minor axis (y for X-main, x for
// Y-main views).  A slice of the main axis is one contiguous slab (scalar
// base, 32-bit lane offsets); the lanes of a wave (consecutive u) read
// neighbouring columns.  As in joseph_fp_column_kernel the sample position is
// clamped to [-2, n], positions outside (-1, n) read only zeros, and a
// sample is one 16-byte load and three lerps.
__global__ void __launch_bounds__(512)
joseph_fp_slab_kernel(const float* __restrict__ gx, const float* __restrict__ gy,
    float* __restrict__ proj, const ProjViewDev* __restrict__ views, VolumeGeom g,
    int nu, int nv, int count, FpStore st)
{
    // the eight waves take one 64-ray row segment of eight consecutive
    // views (nearly coincident rays: the repeats of a sample's cache lines
    // hit the CU's L1; eight measured 7 % faster than four at 512^3 x 720)
    const int u = blockIdx.x * 64 + threadIdx.x;
    const int v = blockIdx.y;
    const int i = blockIdx.z * 8 + threadIdx.y;
    if (i >= count) return;  // whole wave
    const bool pix = u < nu && v < nv;
    const ProjViewDev pv = views[i];
    const AxisInfo ax = axis_info(pv.axis, g);
    const float* base = pv.axis == 0 ? gx : gy;
    JRay r{};
    int lo = 1, hi = 0;
    if (pix && joseph_ray(pv, ax, u, v, r)) joseph_slice_range(r, ax, lo, hi);
    int wlo = lo <= hi ? lo : 0x7fffffff, whi = lo <= hi ? hi : -1;
    for (int off = 32; off > 0; off >>= 1) {
        wlo = min(wlo, __shfl_xor(wlo, off, 64));
        whi = max(whi, __shfl_xor(whi, off, 64));
    }
    wlo = __builtin_amdgcn_readfirstlane(wlo);
    whi = __builtin_amdgcn_readfirstlane(whi);
    const int p1 = ax.n1 + 2 * kJosephGuard;
    const size_t slab_bytes = size_t(ax.n2 + 2 * kJosephGuard - 1) * size_t(p1) * 8u;
    const float f1max = float(ax.n1), f2max = float(ax.n2);
    float acc = 0.f;
    if (wlo > whi) return finish_joseph(proj, i, nu, nv, u, v, pix, lo <= hi, 0.f, r.L, st);
    // the slice coordinate steps by exactly 1 (half-integers below 2^22)
    float c0 = joseph_c0(wlo, ax.n0);
    const char* sl = reinterpret_cast<const char*>(base) + size_t(wlo) * slab_bytes;
    constexpr int kUnroll = 4;
    int s = wlo;
    for (; s + kUnroll - 1 <= whi; s += kUnroll) {
        float4u q[kUnroll];
        float w1[kUnroll], w2[kUnroll];
#pragma unroll
        for (int k = 0; k < kUnroll; ++k) {
            float f1 = joseph_minor(r.a1, r.b1, c0, ax.n1);
            float f2 = joseph_minor(r.a2, r.b2, c0, ax.n2);
            c0 += 1.f;
            f1 = __builtin_amdgcn_fmed3f(f1, -2.f, f1max);
            f2 = __builtin_amdgcn_fmed3f(f2, -2.f, f2max);
            w1[k] = __builtin_amdgcn_fractf(f1);
            w2[k] = __builtin_amdgcn_fractf(f2);
            const int j1 = int(floorf(f1)) + kJosephGuard, j2 = int(floorf(f2)) + kJosephGuard;
            const unsigned o = unsigned(__mul24(j2, p1) + j1) * 8u;
            q[k] = *reinterpret_cast<const float4u*>(sl + o);
            sl += slab_bytes;
        }
#pragma unroll
        for (int k = 0; k < kUnroll; ++k) {
            const float a = fmaf(w1[k], q[k].z - q[k].x, q[k].x);
            const float b = fmaf(w1[k], q[k].w - q[k].y, q[k].y);
            acc += fmaf(w2[k], b - a, a);
        }
    }
    for (; s <= whi; ++s) {
        float f1 = joseph_minor(r.a1, r.b1, c0, ax.n1);
        float f2 = joseph_minor(r.a2, r.b2, c0, ax.n2);
        c0 += 1.f;
        f1 = __builtin_amdgcn_fmed3f(f1, -2.f, f1max);
        f2 = __builtin_amdgcn_fmed3f(f2, -2.f, f2max);
        const float w1 = __builtin_amdgcn_fractf(f1), w2 = __builtin_amdgcn_fractf(f2);
        const int j1 = int(floorf(f1)) + kJosephGuard, j2 = int(floorf(f2)) + kJosephGuard;
        const unsigned o = unsigned(__mul24(j2, p1) + j1) * 8u;
        const float4u q = *reinterpret_cast<const float4u*>(sl + o);
        sl += slab_bytes;
        const float a = fmaf(w1, q.z - q.x, q.x);
        const float b = fmaf(w1, q.w - q.y, q.y);
        acc += fmaf(w2, b - a, a);
    }
    finish_joseph(proj, i, nu, nv, u, v, pix, lo <= hi, acc, r.L, st);
}

// The copy kernels write every entry of their copy, the zero guards among
// them: no zero fill before them (a second pass over the copy; without it one
// OS-SART sweep of 10 subsets at 128 x 128 x 100 x 120 views went from 5.66 to
// 5.32 ms, a SART sweep at 64 x 60 x 48 x 40 views from 2.09 to 1.92 ms).
//
// Z-fastest copy for joseph_fp_column_kernel: [slice][row + guard][z + guard],
// slices along x and rows along y (X-main), or the reverse; 32 x 32 tiles
// through LDS, blockIdx.z is y + guard (X-main) or y (Y-main), blockIdx.x tiles x
// (with its guards for Y-main rows).
template <bool XMAIN>
__global__ void zfast_copy_kernel(const float* __restrict__ in, float* __restrict__ out, int nx, int ny, int nz)
{
    __shared__ float tile[32][33];
    const int x0 = int(blockIdx.x) * 32 - (XMAIN ? 0 : kJosephGuard), e0 = blockIdx.y * 32;
    const int y = int(blockIdx.z) - (XMAIN ? kJosephGuard : 0);
    const int cols = column_pitch(nz);
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int z = e0 + k - kJosephGuard, x = x0 + int(threadIdx.x);
        const bool in_range = x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz;
        tile[k][threadIdx.x] = in_range ? in[(size_t(z) * ny + y) * nx + x] : 0.f;
    }
    __syncthreads();
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int x = x0 + k, e = e0 + threadIdx.x;
        const bool in_range = XMAIN ? x < nx : x < nx + kJosephGuard;
        if (!in_range || e >= cols) continue;
        const size_t slice = XMAIN ? x : y, row = XMAIN ? y + kJosephGuard : x + kJosephGuard;
        const size_t rows = size_t(XMAIN ? ny : nx) + 2 * kJosephGuard;
        out[(slice * rows + row) * cols + e] = tile[threadIdx.x][k];
    }
}

// A volume whose values the Siddon slab projection's differences of taps cannot
// carry (infinities, NaN, values near the type's ends): its copy raises *flag and
// the projection walks instead, which reads only the voxels a ray crosses.
__device__ __forceinline__ void check_value(float v, int* flag)
{
    if (flag && !(fabsf(v) <= 1e37f)) atomicOr(flag, 1);
}

// paired slab copy, X-main: [x][row z + guard][column y + guard];
// blockIdx.z is the row, 32 x 32 (x, column) tiles of the two source planes
// through LDS
__global__ void pair_slab_x_kernel(const float* __restrict__ in, float2* __restrict__ out,
    int nx, int ny, int nz, int* __restrict__ flag)
{
    __shared__ float tile[2][32][33];
    const int r = blockIdx.z;
    const int x0 = blockIdx.x * 32, e0 = blockIdx.y * 32;
    const size_t rows = size_t(nz) + 2 * kJosephGuard - 1, cols = size_t(ny) + 2 * kJosephGuard;
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int y = e0 + k - kJosephGuard, x = x0 + threadIdx.x;
        const bool in_xy = x < nx && y >= 0 && y < ny;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int z = r + h - kJosephGuard;
            tile[h][k][threadIdx.x] = in_xy && z >= 0 && z < nz ? in[(size_t(z) * ny + y) * nx + x] : 0.f;
        }
        check_value(tile[0][k][threadIdx.x], flag);
    }
    __syncthreads();
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int x = x0 + k, e = e0 + threadIdx.x;
        if (x < nx && e < int(cols))
            out[(size_t(x) * rows + r) * cols + e] = make_float2(tile[0][threadIdx.x][k], tile[1][threadIdx.x][k]);
    }
}

// paired slab copy, Y-main: [y][row z + guard][column x + guard] (x stays
// fastest: row copies).  The workgroups are those of the volume's rows, and the
// outer ones write the guard columns beside their own: those of the copy's rows
// have a last one of four columns for 256 (256^3, one tilted view, whole call 115 ->
// 75 us)
__global__ void pair_slab_y_kernel(const float* __restrict__ in, float2* __restrict__ out,
    int nx, int ny, int nz, int* __restrict__ flag)
{
    const int x = blockIdx.x * 256 + threadIdx.x;
    const int y = blockIdx.y, r = blockIdx.z;
    const size_t rows = size_t(nz) + 2 * kJosephGuard - 1, cols = size_t(nx) + 2 * kJosephGuard;
    float2* const row = out + (size_t(y) * rows + r) * cols;
    if (threadIdx.x < kJosephGuard) {
        if (blockIdx.x == 0) row[threadIdx.x] = make_float2(0.f, 0.f);
        if (blockIdx.x == gridDim.x - 1) row[nx + kJosephGuard + threadIdx.x] = make_float2(0.f, 0.f);
    }
    if (x >= nx) return;
    const int z = r - kJosephGuard;
    const float a = z >= 0 && z < nz ? in[(size_t(z) * ny + y) * nx + x] : 0.f;
    const float b = z + 1 >= 0 && z + 1 < nz ? in[(size_t(z + 1) * ny + y) * nx + x] : 0.f;
    row[x + kJosephGuard] = make_float2(a, b);
    check_value(a, flag);
}

// [z][y][x] -> [z][x][y]
__global__ void transpose_xy_kernel(const float* __restrict__ in, float* __restrict__ out,
    int nx, int ny)
{
    __shared__ float tile[32][33];
    const int z = blockIdx.z;
    const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 32;
    const size_t plane = (size_t)nx * ny;
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int y = y0 + k, x = x0 + threadIdx.x;
        if (x < nx && y < ny) tile[k][threadIdx.x] = in[z * plane + (size_t)y * nx + x];
    }
    __syncthreads();
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int x = x0 + k, y = y0 + threadIdx.x;
        if (x < nx && y < ny) out[z * plane + (size_t)x * ny + y] = tile[threadIdx.x][k];
    }
}

// Ray table of the Joseph transpose: the parameters of every ray of `count`
// views, from the same joseph_ray routine the forward kernel calls (so the
// transpose reuses bit-identical lines); L = 0 marks a ray the forward skips.
__global__ void __launch_bounds__(256)
joseph_ray_table_kernel(const ProjViewDev* __restrict__ views, VolumeGeom g, int nu, int nv,
    float4* __restrict__ ab, float* __restrict__ len)
{
    const int u = blockIdx.x * 64 + threadIdx.x;
    const int v = blockIdx.y * 4 + threadIdx.y;
    const int i = blockIdx.z;
    if (u >= nu || v >= nv) return;
    const ProjViewDev pv = views[i];
    const AxisInfo ax = axis_info(pv.axis, g);
    JRay r;
    const size_t k = ((size_t)i * nv + v) * nu + u;
    if (joseph_ray(pv, ax, u, v, r)) {
        ab[k] = make_float4(r.a1, r.b1, r.a2, r.b2);
        len[k] = r.L;
    } else {
        ab[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        len[k] = 0.f;
    }
}

// Joseph transpose: one thread per voxel, gather over views and candidate
// rays.  The candidates of a voxel are the pixels inside the projection of its
// bilinear support on its main-axis slice (FP32 projective map, 0.05 px of
// margin against rounding); each is then tested with the ray's own sample
// position, exactly as the forward kernel computes it.
__global__ void __launch_bounds__(256)
joseph_adjoint_kernel(const float* __restrict__ proj, float* __restrict__ volume,
    const ProjViewDev* __restrict__ views, const float* __restrict__ c32,
    const float4* __restrict__ ray_ab, const float* __restrict__ ray_len, VolumeGeom g,
    int nu, int nv, int count, int accumulate)
{
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    const int z = blockIdx.z;
    if (x >= g.nx || y >= g.ny) return;
    const float margin = 0.05f;
    float acc = 0.f;
    for (int i = 0; i < count; ++i) {
        const ProjViewDev pv = views[i];
        const AxisInfo ax = axis_info(pv.axis, g);
        const int s = pick(ax.p0, x, y, z), i1 = pick(ax.p1, x, y, z), i2 = pick(ax.p2, x, y, z);
        const float* c = c32 + (size_t)i * 12;
        // world coordinates of the main-axis plane and of the minor neighbours
        const float m0 = pick(ax.p0, g.ox, g.oy, g.oz) + float(s) * pick(ax.p0, g.vx, g.vy, g.vz);
        const float o1 = pick(ax.p1, g.ox, g.oy, g.oz), w1 = pick(ax.p1, g.vx, g.vy, g.vz);
        const float o2 = pick(ax.p2, g.ox, g.oy, g.oz), w2 = pick(ax.p2, g.vx, g.vy, g.vz);
        float umin = 1e30f, umax = -1e30f, vmin = 1e30f, vmax = -1e30f;
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float m1 = o1 + float(i1 + ((k & 1) ? 1 : -1)) * w1;
            const float m2 = o2 + float(i2 + ((k & 2) ? 1 : -1)) * w2;
            float p[3];
            p[0] = ax.p0 == 0 ? m0 : (ax.p1 == 0 ? m1 : m2);
            p[1] = ax.p0 == 1 ? m0 : (ax.p1 == 1 ? m1 : m2);
            p[2] = ax.p0 == 2 ? m0 : (ax.p1 == 2 ? m1 : m2);
            const float den = c[8] * p[0] + c[9] * p[1] + c[10] * p[2] + c[11];
            if (!(den > 1e-6f)) { ok = false; break; }
            const float rd = 1.f / den;
            const float uu = (c[0] * p[0] + c[1] * p[1] + c[2] * p[2] + c[3]) * rd;
            const float vv = (c[4] * p[0] + c[5] * p[1] + c[6] * p[2] + c[7]) * rd;
            umin = fminf(umin, uu); umax = fmaxf(umax, uu);
            vmin = fminf(vmin, vv); vmax = fmaxf(vmax, vv);
        }
        if (!ok) continue;
        const int ulo = max(0, int(ceilf(umin - margin)));
        const int uhi = min(nu - 1, int(floorf(umax + margin)));
        const int vlo = max(0, int(ceilf(vmin - margin)));
        const int vhi = min(nv - 1, int(floorf(vmax + margin)));
        const size_t vb = (size_t)i * nu * nv;
        const float* pi = proj + vb;
        const float4* abi = ray_ab + vb;
        const float* li = ray_len + vb;
        for (int vv = vlo; vv <= vhi; ++vv)
            for (int uu = ulo; uu <= uhi; ++uu) {
                const size_t k = (size_t)vv * nu + uu;
                // The candidate test is branch-free, so the three loads issue
                // at once (a skip after the first load made them wait in
                // turn); a rejected candidate leaves the sum as it is.
                const float L = li[k];
                const float4 a = abi[k];
                const float py = pi[k];
                JRay r;
                r.a1 = a.x; r.b1 = a.y; r.a2 = a.z; r.b2 = a.w; r.L = L;
                float f1, f2;
                joseph_sample(r, ax, s, f1, f2);
                const float g1 = floorf(f1), g2 = floorf(f2);
                const float w1 = f1 - g1, w2 = f2 - g2;
                // the voxel is tap j or j + 1 of the ray's sample on each axis
                const bool a0 = float(i1) == g1, a1 = float(i1) == g1 + 1.f;
                const bool b0 = float(i2) == g2, b1 = float(i2) == g2 + 1.f;
                const float wa = a0 ? 1.f - w1 : w1, wb = b0 ? 1.f - w2 : w2;
                const float t = fmaf(py * L, wa * wb, acc);
                acc = (L != 0.f && (a0 || a1) && (b0 || b1)) ? t : acc;
            }
    }
    float* dst = volume + ((size_t)z * g.ny + y) * g.nx + x;
    *dst = accumulate ? *dst + acc : acc;
}

// ---------------------------------------------------------------------------
// Siddon
// ---------------------------------------------------------------------------
// Exact Amanatides-Woo walk of one ray through the [z][y][x] volume, clipped
// to t in [0, 1] and to the volume box.  Plane crossings are recomputed from
// integer indices as (plane - src) * (1 / ray), and the ray sum adds the
// segments in walk order.  (For a ray outside the upper faces: the caller asks
// siddon_in_upper_face, whose FP64 registers the slab kernel's loop has no room
// for.)
__device__ __forceinline__ float siddon_walk(const float* __restrict__ vol, const SiddonViewDev& sv, const VolumeGeom& g,
    int u, int v)
{
    float src[3], ray[3];
    siddon_ray_geom(sv, u, v, src, ray);
    const Box b = volume_box(g);
    const int dims[3] = { g.nx, g.ny, g.nz };
    const float vox[3] = { g.vx, g.vy, g.vz };
    float t0, t1, acc = 0.f;
    if (!clip_ray(src, ray, b.lo, b.hi, t0, t1)) return 0.f;
    const float len = sqrtf(ray[0] * ray[0] + ray[1] * ray[1] + ray[2] * ray[2]);
    int idx[3], step[3];
    float tn[3], rcp[3];
    bool valid[3];
    for (int k = 0; k < 3; ++k) {
        const float e = src[k] + t0 * ray[k];
        idx[k] = min(dims[k] - 1, max(0, int(floorf((e - b.lo[k]) / vox[k]))));
        step[k] = ray[k] >= 0.f ? 1 : -1;
        valid[k] = fabsf(ray[k]) > 1e-8f;
        rcp[k] = valid[k] ? 1.f / ray[k] : 0.f;
        const float plane = b.lo[k] + float(idx[k] + (step[k] > 0 ? 1 : 0)) * vox[k];
        tn[k] = valid[k] ? (plane - src[k]) * rcp[k] : 3.0e38f;
    }
    float t = t0;
    const int max_steps = g.nx + g.ny + g.nz + 3;
    for (int n = 0; n < max_steps && t < t1; ++n) {
        const float tnext = fminf(fminf(tn[0], tn[1]), fminf(tn[2], t1));
        acc += vol[((size_t)idx[2] * g.ny + idx[1]) * g.nx + idx[0]] * (tnext - t);
        t = tnext;
        int k;
        if (tn[0] <= tn[1] && tn[0] <= tn[2]) k = 0;
        else if (tn[1] <= tn[2]) k = 1;
        else k = 2;
        idx[k] += step[k];
        if (idx[k] < 0 || idx[k] >= dims[k]) break;
        const float plane = b.lo[k] + float(idx[k] + (step[k] > 0 ? 1 : 0)) * vox[k];
        tn[k] = (plane - src[k]) * rcp[k];
    }
    return acc * len;
}

// The projections of a volume of ones, the algebraic solvers' row weights, in
// closed form: no volume, copies or gathers.
//
// Joseph: a slice adds the weights of its taps inside the volume, the product
// over both minor axes of min(f + 1, n - f) clamped to [0, 1].  It is 1 in every
// slice where the ray lies inside [0, n - 1] on both axes, so only the slices at
// the ends (and one more on either side) are evaluated.
// (OS-SART of 10 subsets at 128 x 128 x 100 x 120 views of 256 x 192: 1.65 ms
// with the projection of a volume of ones, 350 us with its copies, 1.36 here.)
__global__ void __launch_bounds__(256)
joseph_ones_kernel(float* __restrict__ proj, const ProjViewDev* __restrict__ views, VolumeGeom g, int nu, int nv)
{
    const int u = blockIdx.x * 64 + threadIdx.x;
    const int v = blockIdx.y * 4 + threadIdx.y;
    const int i = blockIdx.z;
    if (u >= nu || v >= nv) return;
    const ProjViewDev pv = views[i];
    const AxisInfo ax = axis_info(pv.axis, g);
    JRay r{};
    int lo = 1, hi = 0;
    if (joseph_ray(pv, ax, u, v, r)) joseph_slice_range(r, ax, lo, hi);
    // slices inside on both axes
    float slo = float(lo), shi = float(hi);
    const float h0 = 0.5f * float(ax.n0 - 1);
    const float a[2] = { r.a1, r.a2 }, n[2] = { float(ax.n1), float(ax.n2) };
    const float b[2] = { r.b1 + 0.5f * float(ax.n1 - 1), r.b2 + 0.5f * float(ax.n2 - 1) };
    for (int k = 0; k < 2; ++k) {
        if (fabsf(a[k]) > 1e-12f) {
            const float t0 = -b[k] / a[k] + h0, t1 = (n[k] - 1.f - b[k]) / a[k] + h0;
            slo = fmaxf(slo, fminf(t0, t1));
            shi = fminf(shi, fmaxf(t0, t1));
        } else if (!(b[k] >= 0.f && b[k] <= n[k] - 1.f)) {
            shi = -1.f;
        }
    }
    const int ilo = int(ceilf(fminf(slo, float(hi)))) + 1, ihi = int(floorf(fmaxf(shi, -1.f))) - 1;
    float sum = ilo <= ihi ? float(ihi - ilo + 1) : 0.f;
    for (int s = lo; s <= hi; ++s) {
        if (s == ilo && ilo <= ihi) s = ihi + 1;  // (<= hi: shi and a slice less)
        float f1, f2;
        joseph_sample(r, ax, s, f1, f2);
        sum += __builtin_amdgcn_fmed3f(fminf(f1 + 1.f, n[0] - f1), 0.f, 1.f) *
            __builtin_amdgcn_fmed3f(fminf(f2 + 1.f, n[1] - f2), 0.f, 1.f);
    }
    proj[((size_t)i * nv + v) * nu + u] = sum * r.L;
}

// Siddon: the length of the ray inside the volume, between the ends the walk
// clips it to
__global__ void __launch_bounds__(256)
siddon_ones_kernel(float* __restrict__ proj, const SiddonViewDev* __restrict__ views, VolumeGeom g, int nu, int nv)
{
    const int u = blockIdx.x * 64 + threadIdx.x;
    const int v = blockIdx.y * 4 + threadIdx.y;
    const int i = blockIdx.z;
    if (u >= nu || v >= nv) return;
    float src[3], ray[3], t0, t1;
    siddon_ray_geom(views[i], u, v, src, ray);
    const Box b = volume_box(g);
    const bool hit = clip_ray(src, ray, b.lo, b.hi, t0, t1) && !siddon_in_upper_face(views[i], g, u, v);
    const float len = sqrtf(ray[0] * ray[0] + ray[1] * ray[1] + ray[2] * ray[2]);
    proj[((size_t)i * nv + v) * nu + u] = hit ? (t1 - t0) * len : 0.f;
}

// Siddon projection by the walk, one lane per ray.  It serves the plans whose
// rays are too few to pay for the volume copies of siddon_fp_slab_kernel.
__global__ void __launch_bounds__(256)
siddon_fp_kernel(const float* __restrict__ vol, float* __restrict__ proj,
    const SiddonViewDev* __restrict__ views, VolumeGeom g, int nu, int nv, int count, int accumulate)
{
    // a workgroup is an 8 x 4 pixel tile of eight consecutive views: their
    // rays nearly coincide, so the scattered voxel reads of the walk share
    // cache lines in the CU's L1
    const int u = blockIdx.x * 8 + (threadIdx.x & 7);
    const int v = blockIdx.y * 4 + ((threadIdx.x >> 3) & 3);
    const int i = int(blockIdx.z) * 8 + int(threadIdx.x >> 5);
    if (u >= nu || v >= nv || i >= count) return;
    const SiddonViewDev& sv = views[i];
    const float acc = siddon_in_upper_face(sv, g, u, v) ? 0.f : siddon_walk(vol, sv, g, u, v);
    float* dst = proj + ((size_t)i * nv + v) * nu + u;
    *dst = accumulate ? *dst + acc : acc;
}

__global__ void clear_flag_kernel(int* __restrict__ flag) { *flag = 0; }

// One minor axis of a ray in cell coordinates (cell j spans [j, j + 1)) over
// the slabs of its main axis: in slab c it runs from low to low + |slope|,
// low = slope (c - n0 / 2) + base, so at |slope| <= 1 it crosses at most one
// plane, and the part of the slab it spends past it is
// clamp((fract(low) + |slope| - 1) / |slope|).
struct SiddonMinor {
    float slope, base;  // of low
    float inv, off;     // 1 / |slope|, (|slope| - 1) / |slope|
};

__device__ __forceinline__ SiddonMinor siddon_minor(double at_mid, double slope, int n, int n0, int plane)
{
    SiddonMinor m;
    if (siddon_stays(slope, n, 1.0, n0)) {
        slope = 0.0;
        if (plane >= 0) at_mid = double(plane);
    }
    m.slope = float(slope);
    m.base = float(at_mid + fmin(slope, 0.0));
    const float a = fabsf(m.slope);
    m.inv = a > 1e-30f ? 1.f / a : 1e30f;
    m.off = fminf(a * m.inv, 1.f) - m.inv;
    return m;
}

// slabs in which the axis can lie inside [0, n), with a slab of margin
__device__ __forceinline__ void siddon_slab_range(const SiddonMinor& m, float half0, int n, float& lo, float& hi)
{
    const float a = fabsf(m.slope);
    if (a > 1e-12f) {
        const float r = 1.f / m.slope;
        const float t0 = (-a - m.base) * r + half0, t1 = (float(n) - m.base) * r + half0;
        lo = fmaxf(lo, fminf(t0, t1) - 1.f);
        hi = fminf(hi, fmaxf(t0, t1) + 1.f);
    } else if (m.base < -1.f || m.base > float(n)) {
        hi = -1.f;
    }
}

// Siddon projection over slabs: a ray whose main axis (the largest |ray /
// voxel| of X and Y, per ray) advances one slab at a time crosses at most one
// plane of either minor axis inside it, so the up to three voxels it visits
// lie in one 2 x 2 block of taps and their segments follow from two clamped
// fractions: h1, h2 (the parts of the slab past the crossing of either axis)
// and the part past both.  With the paired slab copies of the Joseph
// projection a slab is one 16-byte load, where the walk took a dependent
// 4-byte gather and ~50 instructions for each of ~1.5 voxels.
// Bound: one 16-cycle gather and ~75 VALU cycles (on four SIMDs) a slab, both
// about 18 cycles a wave on each CU.  256^3 x 360 views of 512 x 384, copies
// included: 27.7 ms by the walk -> 10.5 ms here (10.8 with a tilted detector);
// 240 x 231 x 190 x 240 views of 480 x 360, tilted: 12.4 -> 6.0 ms.
// The ray is set up in FP64 about the middle of the volume, so positions carry
// ~1e-5 voxel of rounding.  Rays that the slab form does not cover (steepest
// along Z, or the source or the pixel inside the main-axis extent, where t in
// [0, 1] can clip) walk, as do all rays of a flagged volume.  A call whose rays all
// have one main axis comes with that axis's copy alone.
__global__ void __launch_bounds__(512)
siddon_fp_slab_kernel(const float* __restrict__ gx, const float* __restrict__ gy, const float* __restrict__ vol,
    const int* __restrict__ flag, float* __restrict__ proj, const SiddonViewDev* __restrict__ views, VolumeGeom g,
    int nu, int nv, int count, int accumulate)
{
    // eight waves: one 64-ray row segment of eight consecutive views, as in
    // joseph_fp_slab_kernel
    const int u = blockIdx.x * 64 + threadIdx.x;
    const int v = blockIdx.y;
    const int i = blockIdx.z * 8 + threadIdx.y;
    if (i >= count) return;  // whole wave
    const bool pix = u < nu;
    const SiddonViewDev sv = views[i];
    const bool face = siddon_in_upper_face(sv, g, u, v);
    double S[3], R[3], r[3], len2 = 0.0;
    siddon_ray_geom(sv, u, v, r);
    const double lo[3] = { double(g.ox) - 0.5 * double(g.vx), double(g.oy) - 0.5 * double(g.vy),
                           double(g.oz) - 0.5 * double(g.vz) };
    const double vox[3] = { double(g.vx), double(g.vy), double(g.vz) };
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        len2 += r[k] * r[k];
        S[k] = (double(sv.src[k]) - lo[k]) / vox[k];
        R[k] = r[k] / vox[k];
    }
    const bool ymain = !(fabs(R[0]) >= fabs(R[1]));
    const double r0 = ymain ? R[1] : R[0], s0 = ymain ? S[1] : S[0];
    const double r1 = ymain ? R[0] : R[1], s1 = ymain ? S[0] : S[1];
    const int n0 = ymain ? g.ny : g.nx, n1 = ymain ? g.nx : g.ny, n2 = g.nz;
    const double rc = 1.0 / r0;
    const double ta = -s0 * rc, tb = (double(n0) - s0) * rc;
    const bool slabs = fabs(R[2]) <= fabs(r0) && fmin(ta, tb) >= 0.0 && fmax(ta, tb) <= 1.0 && (ymain ? gy : gx) && *flag == 0;
    const double mid = 0.5 * double(n0) - s0;
    const SiddonMinor m1 = siddon_minor(s1 + mid * (r1 * rc), r1 * rc, n1, n0, ymain ? sv.plane[0] : sv.plane[1]);
    const SiddonMinor m2 = siddon_minor(S[2] + mid * (R[2] * rc), R[2] * rc, n2, n0, sv.plane[2]);
    const float len = float(sqrt(len2) * fabs(rc));
    const float half0 = 0.5f * float(n0);
    float flo = 0.f, fhi = float(n0 - 1);
    siddon_slab_range(m1, half0, n1, flo, fhi);
    siddon_slab_range(m2, half0, n2, flo, fhi);
    const bool live = pix && slabs && flo <= fhi;
    const int clo = live ? int(flo) : 0x7fffffff, chi = live ? int(fhi) : -1;
    // past both crossings: the slopes agree in sign -> min(h1, h2), else
    // h1 - min(h1, 1 - h2): with y = sa h2 + sb and m = min(h1, y), sa m + sb h1
    const bool agree = (m1.slope < 0.f) == (m2.slope < 0.f);
    const float sa = agree ? 1.f : -1.f, sb = agree ? 0.f : 1.f;
    float acc = 0.f;
    // waves near a diagonal hold rays of both main axes: one pass for each
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        const bool mine = live && ymain == (pass == 1);
        if (!__any(mine)) continue;
        int wlo = mine ? clo : 0x7fffffff, whi = mine ? chi : -1;
        for (int off = 32; off > 0; off >>= 1) {
            wlo = min(wlo, __shfl_xor(wlo, off, 64));
            whi = max(whi, __shfl_xor(whi, off, 64));
        }
        wlo = __builtin_amdgcn_readfirstlane(wlo);
        whi = __builtin_amdgcn_readfirstlane(whi);
        if (!mine) continue;
        const int p1 = (pass ? g.nx : g.ny) + 2 * kJosephGuard;
        const size_t slab_bytes = size_t(n2 + 2 * kJosephGuard - 1) * size_t(p1) * 8u;
        const float top1 = float(pass ? g.nx : g.ny), top2 = float(n2);
        const char* sl = reinterpret_cast<const char*>(pass ? gy : gx) + size_t(wlo) * slab_bytes;
        float c = float(wlo) - half0;  // exact half-integers
        auto taps = [&](float& h1, float& h2) {
            const float f1 = fmaf(m1.slope, c, m1.base), f2 = fmaf(m2.slope, c, m2.base);
            c += 1.f;
            const float g1 = floorf(f1), g2 = floorf(f2);
            h1 = __builtin_amdgcn_fmed3f(fmaf(f1 - g1, m1.inv, m1.off), 0.f, 1.f);
            h2 = __builtin_amdgcn_fmed3f(fmaf(f2 - g2, m2.inv, m2.off), 0.f, 1.f);
            // outside [-1, n] both taps of an axis are guards
            const int j1 = int(__builtin_amdgcn_fmed3f(g1, -2.f, top1)) + kJosephGuard;
            const int j2 = int(__builtin_amdgcn_fmed3f(g2, -2.f, top2)) + kJosephGuard;
            const float4u q = *reinterpret_cast<const float4u*>(sl + unsigned(__mul24(j2, p1) + j1) * 8u);
            sl += slab_bytes;
            return q;
        };
        auto sum = [&](const float4u& q, float h1, float h2) {
            const float m = fminf(h1, fmaf(sa, h2, sb));
            const float w = fmaf(sa, m, sb * h1);
            // q: (j2, j1), (j2 + 1, j1), (j2, j1 + 1), (j2 + 1, j1 + 1)
            const float d2 = q.y - q.x, d1 = q.z - q.x;
            const float both = (q.w - q.y) - d1;
            acc += fmaf(w, both, fmaf(h2, d2, fmaf(h1, d1, q.x)));
        };
        int s = wlo;
        constexpr int kUnroll = 4;
        for (; s + kUnroll - 1 <= whi; s += kUnroll) {
            float4u q[kUnroll];
            float h1[kUnroll], h2[kUnroll];
#pragma unroll
            for (int k = 0; k < kUnroll; ++k) q[k] = taps(h1[k], h2[k]);
#pragma unroll
            for (int k = 0; k < kUnroll; ++k) sum(q[k], h1[k], h2[k]);
        }
        for (; s <= whi; ++s) {
            float h1, h2;
            const float4u q = taps(h1, h2);
            sum(q, h1, h2);
        }
    }
    if (!pix) return;
    const float out = slabs ? acc * len : face ? 0.f : siddon_walk(vol, sv, g, u, v);
    float* dst = proj + ((size_t)i * nv + v) * nu + u;
    *dst = accumulate ? *dst + out : out;
}

// Siddon transpose: one thread per voxel; for each view the candidate rays
// are the pixels inside the projection of the voxel cube, and each candidate
// contributes y * |segment inside the cube, clipped like the forward walk|.
__global__ void __launch_bounds__(256)
siddon_adjoint_kernel(const float* __restrict__ proj, float* __restrict__ volume,
    const SiddonViewDev* __restrict__ views, const float* __restrict__ c32, VolumeGeom g,
    int nu, int nv, int count, int accumulate)
{
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    const int z = blockIdx.z;
    if (x >= g.nx || y >= g.ny) return;
    const Box b = volume_box(g);
    float clo[3], chi[3];  // the voxel's cube
    clo[0] = b.lo[0] + float(x) * g.vx; chi[0] = b.lo[0] + float(x + 1) * g.vx;
    clo[1] = b.lo[1] + float(y) * g.vy; chi[1] = b.lo[1] + float(y + 1) * g.vy;
    clo[2] = b.lo[2] + float(z) * g.vz; chi[2] = b.lo[2] + float(z + 1) * g.vz;
    const float margin = 0.05f;
    const bool surface = x == 0 || x == g.nx - 1 || y == 0 || y == g.ny - 1 || z == 0 || z == g.nz - 1;
    float acc = 0.f;
    for (int i = 0; i < count; ++i) {
        // candidate pixels: the projected box of the voxel's 8 corners (FP32
        // map; the 0.05 px margin covers its rounding, and every candidate
        // is then tested with its own segment)
        const float* c = c32 + (size_t)i * 12;
        float umin = 3.0e38f, umax = -3.0e38f, vmin = 3.0e38f, vmax = -3.0e38f;
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float X = (k & 1) ? chi[0] : clo[0];
            const float Y = (k & 2) ? chi[1] : clo[1];
            const float Z = (k & 4) ? chi[2] : clo[2];
            const float den = c[8] * X + c[9] * Y + c[10] * Z + c[11];
            ok = ok && den > 1e-6f;
            const float rd = __builtin_amdgcn_rcpf(den);
            const float uu = proj_coord(c, 0, X, Y, Z, rd), vv = proj_coord(c, 4, X, Y, Z, rd);
            umin = fminf(umin, uu); umax = fmaxf(umax, uu);
            vmin = fminf(vmin, vv); vmax = fmaxf(vmax, vv);
        }
        if (!ok) continue;
        const int ulo = max(0, int(ceilf(umin - margin)));
        const int uhi = min(nu - 1, int(floorf(umax + margin)));
        const int vlo = max(0, int(ceilf(vmin - margin)));
        const int vhi = min(nv - 1, int(floorf(vmax + margin)));
        if (ulo > uhi || vlo > vhi) continue;
        const SiddonViewDev sv = views[i];
        const float* pi = proj + (size_t)i * nu * nv;
        for (int vv = vlo; vv <= vhi; ++vv)
            for (int uu = ulo; uu <= uhi; ++uu) {
                float src[3], ray[3];
                siddon_ray_geom(sv, uu, vv, src, ray);
                // the voxel's interval from the forward walk's own plane
                // crossings; the volume clip (whose faces are a voxel or more
                // away from an interior voxel's) binds only on the surface
                float a = -3.0e38f, e = 3.0e38f;
                cell_interval(src[0], ray[0], b.lo[0], g.vx, x, g.nx, a, e);
                cell_interval(src[1], ray[1], b.lo[1], g.vy, y, g.ny, a, e);
                cell_interval(src[2], ray[2], b.lo[2], g.vz, z, g.nz, a, e);
                if (!(e > a)) continue;
                if (surface) {
                    float t0, t1;
                    if (!clip_ray(src, ray, b.lo, b.hi, t0, t1) || siddon_in_upper_face(sv, g, uu, vv)) continue;
                    a = fmaxf(a, t0);
                    e = fminf(e, t1);
                } else {
                    a = fmaxf(a, 0.f);
                    e = fminf(e, 1.f);
                }
                if (!(e > a)) continue;
                const float len = sqrtf(ray[0] * ray[0] + ray[1] * ray[1] + ray[2] * ray[2]);
                acc += pi[(size_t)vv * nu + uu] * ((e - a) * len);
            }
    }
    float* dst = volume + ((size_t)z * g.ny + y) * g.nx + x;
    *dst = accumulate ? *dst + acc : acc;
}

// Operator-form FDK backprojections, the iterative B of the reference's
// automatic flat selection (fdk_bp_kernel_fdk_weight_v2 and
// fdk_bp_kernel_matched_weight, src/FlatFpBp/BP/kernels/YkBpFdkKernel.cu:228-466):
// unfiltered views, exact bilinear sample at the projected voxel centre (zero
// outside the detector), per-sample weight
//   FDK:     SOD^2 dtheta fscale / (Cc . [X, 1])^2,  Cc = (-src / SOD, SOD)
//   matched: L^3 / (|X - src|^2 SDD_plane) * vx vy vz / (du dv),
//            L^2 = |detS + u detU + v detV - src|^2;
//   voxel-driven Joseph (joseph_bp_v3_kernel,
//   src/FlatFpBp/BP/kernels/YkBPJosephKernel.cu:624-735): the physical length
//   of X - src through one voxel along its main axis m = argmax |d_k / v_k|
//   (ties X, then Y): v_m |d| / |d_m|.
constexpr int kOpBpZ = 8;
constexpr int kOpBpShortZ = 2;
// zero pixels before and after a paired view's rows and columns: two, as both
// taps of a sample clamped off the detector must be zeros (one zero and one pixel
// of weight zero would spread a pixel that is not finite)
constexpr int kViewGuard = 2;
// entries of a paired view's row, and its rows (the last one pairs with zeros)
__host__ __device__ __forceinline__ int paired_pitch(int nu) { return nu + 2 * kViewGuard; }
__host__ __device__ __forceinline__ int paired_rows(int nv) { return nv + 2 * kViewGuard - 1; }
enum OpBpMode { kOpFdk = 0, kOpMatched = 1, kOpJosephVoxel = 2 };

__device__ __forceinline__ float bilinear_view(const float* __restrict__ p, int nu, int nv, float u, float v)
{
    const float fu = floorf(u), fv = floorf(v);
    const int iu = int(fu), iv = int(fv);
    const float a = u - fu, b = v - fv;
    const bool u0 = iu >= 0 && iu < nu, u1 = iu + 1 >= 0 && iu + 1 < nu;
    const bool v0 = iv >= 0 && iv < nv, v1 = iv + 1 >= 0 && iv + 1 < nv;
    const float t00 = (u0 && v0) ? p[(size_t)iv * nu + iu] : 0.f;
    const float t01 = (u1 && v0) ? p[(size_t)iv * nu + iu + 1] : 0.f;
    const float t10 = (u0 && v1) ? p[(size_t)(iv + 1) * nu + iu] : 0.f;
    const float t11 = (u1 && v1) ? p[(size_t)(iv + 1) * nu + iu + 1] : 0.f;
    return (1.f - b) * ((1.f - a) * t00 + a * t01) + b * ((1.f - a) * t10 + a * t11);
}

// square root to half an ulp for a normal x > 0: one Newton step on the
// hardware's reciprocal root (16 cycles, the library's scaled form takes ~40)
__device__ __forceinline__ float op_sqrt(float x)
{
    const float r = __builtin_amdgcn_rsqf(x), s = x * r;
    return fmaf(fmaf(-s, s, x), 0.5f * r, s);
}

// the part of a view's sample weight that a voxel column shares
template <int MODE>
struct OpColumn {
    float xy2, inv, base;  // |X - src|^2 in the plane; 1 / main-axis steps (Joseph); FDK denominator at Z = 0
    bool zmain;            // some lane of the wave may have main axis Z (Joseph)

    __device__ __forceinline__ OpColumn(const OpBpViewDev& c, const VolumeGeom& g, float X, float Y, float Za, float Zb)
    {
        const float dx = X - c.src[0], dy = Y - c.src[1];
        xy2 = dx * dx + dy * dy;
        inv = base = 0.f;
        zmain = false;
        if constexpr (MODE == kOpJosephVoxel) {
            base = fmaxf(fabsf(dx / g.vx), fabsf(dy / g.vy));
            inv = __builtin_amdgcn_rcpf(base);
            zmain = __any(!(fmaxf(fabsf(Za - c.src[2]), fabsf(Zb - c.src[2])) <= base * g.vz));
        } else if constexpr (MODE == kOpFdk) {
            base = c.cc[0] * X + c.cc[1] * Y + c.cc[3];
        }
    }

    // weight of the sample at (u, v) of the column's voxel at height Z; `ok`
    // is cleared when it adds nothing
    __device__ __forceinline__ float weight(const OpBpViewDev& c, float ivz, float scale, float Z, float u, float v,
        bool& ok) const
    {
        if constexpr (MODE == kOpJosephVoxel) {
            // v_m |d| / |d_m|, m the axis of the largest |d_k / v_k|
            const float dz = Z - c.src[2];
            const float len = op_sqrt(fmaf(dz, dz, xy2));
            return zmain ? len * __builtin_amdgcn_rcpf(fmaxf(base, fabsf(dz * ivz))) : len * inv;
        } else if constexpr (MODE == kOpMatched) {
            const float L2 = c.l2[0] + u * (c.l2[1] + u * c.l2[3]) + v * (c.l2[2] + u * c.l2[4] + v * c.l2[5]);
            const float dz = Z - c.src[2], lsq = fmaf(dz, dz, xy2);
            ok = ok && L2 >= 1e-8f && lsq >= 1e-8f;
            return L2 * op_sqrt(L2) * __builtin_amdgcn_rcpf(lsq) * c.inv_sdd_plane * scale;
        } else {
            const float cn = fmaf(c.cc[2], Z, base);
            const float rc = __builtin_amdgcn_rcpf(cn);
            ok = ok && fabsf(cn) >= 1e-8f;
            return c.wbase * rc * rc;
        }
    }
};

// One lane per (x, y) column of kOpBpZ voxels.
// PAIRED: the samples come from a paired guarded copy of the views
// (pair_views_kernel), one 16-byte load each at a position clamped into the
// copy, with no bounds branches; the loads of kOpBatch slices are issued
// together.  Otherwise four bounds-checked taps of the views themselves.
// FRONT: every voxel (and the run's overhang past the last slice) lies before
// the source of every view with a weight that is not singular, so no sample is
// tested.
// Bound of the paired form: about 100 VALU cycles (25 a CU) and one 16-cycle
// gather a sample.  256^3 x 360 views of 512 x 384, four taps -> paired: FDK
// 10.2 -> 4.4 ms, pseudo-matched 11.4 -> 6.1, voxel-driven Joseph 11.1 -> 5.9,
// the copy included.
// A launch serves one unit of views or, with `units`, a volume for each of
// several; view_step 0 gives every view the first one's pixels: the column
// weights of all subsets of a solver are one launch, and its update is made by
// the store (SART at 64 x 60 x 48 x 40 single views 1.26 -> 0.80 ms, OS-SART of
// 10 subsets at 128 x 128 x 100 x 120 views 1.86 -> 1.65 ms).
constexpr int kOpBatch = 4;
template <int MODE, bool PAIRED, bool FRONT, int ZR>
__global__ void __launch_bounds__(256)
fdk_operator_bp_kernel(const float* __restrict__ proj, float* __restrict__ volume,
    const OpBpViewDev* __restrict__ views, VolumeGeom g, int nu, int nv, int count, float scale,
    int view_step, const OpBpUnit* __restrict__ units, int z_blocks, OpBpStore st)
{
    const int x = blockIdx.x * 16 + int(threadIdx.x % 16);
    const int y = blockIdx.y * 16 + int(threadIdx.x / 16);
    int z_block = int(blockIdx.z);
    if (units) {
        const int k = z_block / z_blocks;
        z_block -= k * z_blocks;
        const OpBpUnit unit = units[k];
        views += unit.first;
        count = unit.count;
        scale = unit.scale;
        volume += (size_t)k * g.nz * g.ny * g.nx;
    }
    const int z0 = z_block * ZR;
    if (x >= g.nx || y >= g.ny) return;
    const float X = g.ox + x * g.vx, Y = g.oy + y * g.vy;
    const float Za = g.oz + z0 * g.vz, Zb = g.oz + (z0 + ZR - 1) * g.vz;
    constexpr int kBatch = ZR < kOpBatch ? ZR : kOpBatch;
    float acc[ZR];
#pragma unroll
    for (int k = 0; k < ZR; ++k) acc[k] = 0.f;
    const float ivz = 1.f / g.vz;
    const int pitch = paired_pitch(nu), rows = paired_rows(nv);
#pragma unroll 1
    for (int i = 0; i < count; ++i) {
        const OpBpViewDev& c = views[i];
        const OpColumn<MODE> col(c, g, X, Y, Za, Zb);
        // the view's map at this voxel column; each slice adds its Z term
        const float d0 = fmaf(c.cd[1], Y, fmaf(c.cd[0], X, c.cd[3]));
        const float u0 = fmaf(c.cu[1], Y, fmaf(c.cu[0], X, c.cu[3]));
        const float v0 = fmaf(c.cv[1], Y, fmaf(c.cv[0], X, c.cv[3]));
        // numerators of u and v and the reciprocal depth at slice k: one
        // Newton step on the hardware reciprocal brings u and v within an ulp
        // or so of the quotients (the sample position is the sensitive
        // input), for two FMAs instead of two divisions
        auto project = [&](int k, float& Z, float& un, float& vn, float& rd) {
            Z = g.oz + (z0 + k) * g.vz;
            const float den = fmaf(c.cd[2], Z, d0);
            rd = __builtin_amdgcn_rcpf(den);
            rd = fmaf(rd, fmaf(-den, rd, 1.f), rd);
            un = fmaf(c.cu[2], Z, u0);
            vn = fmaf(c.cv[2], Z, v0);
            return den >= 1e-8f;
        };
        if constexpr (PAIRED) {
            const char* p = reinterpret_cast<const char*>(proj) + size_t(i * view_step) * rows * pitch * 8u;
            constexpr float kGuard = float(kViewGuard);
            const float umax = float(nu) + kGuard, vmax = float(nv) + kGuard;
            const unsigned row_bytes = unsigned(pitch) * 8u;
#pragma unroll
            for (int k0 = 0; k0 < ZR; k0 += kBatch) {
                float4u q[kBatch];
                float a[kBatch], b[kBatch], w[kBatch];
                bool on[kBatch];
#pragma unroll
                for (int k = 0; k < kBatch; ++k) {
                    float Z, un, vn, rd;
                    on[k] = project(k0 + k, Z, un, vn, rd);
                    w[k] = col.weight(c, ivz, scale, Z, un * rd, vn * rd, on[k]);
                    // positions in the copy (pixel + guard); a clamped sample
                    // lies on guards only
                    const float u = __builtin_amdgcn_fmed3f(fmaf(un, rd, kGuard), 0.f, umax);
                    const float v = __builtin_amdgcn_fmed3f(fmaf(vn, rd, kGuard), 0.f, vmax);
                    a[k] = __builtin_amdgcn_fractf(u);
                    b[k] = __builtin_amdgcn_fractf(v);
                    q[k] = *reinterpret_cast<const float4u*>(p + (__umul24(unsigned(int(v)), row_bytes) + unsigned(int(u)) * 8u));
                }
#pragma unroll
                for (int k = 0; k < kBatch; ++k) {
                    // q: (row, col), (row + 1, col), (row, col + 1), (row + 1, col + 1)
                    const float a0 = 1.f - a[k], b0 = 1.f - b[k];
                    const float s = fmaf(b[k], fmaf(a[k], q[k].w, a0 * q[k].y), b0 * fmaf(a[k], q[k].z, a0 * q[k].x));
                    const float t = fmaf(s, w[k], acc[k0 + k]);
                    acc[k0 + k] = FRONT || on[k] ? t : acc[k0 + k];
                }
            }
        } else {
            const float* p = proj + (size_t)(i * view_step) * nu * nv;
#pragma unroll
            for (int k = 0; k < ZR; ++k) {
                if (z0 + k >= g.nz) break;
                float Z, un, vn, rd;
                bool ok = project(k, Z, un, vn, rd);
                const float u = un * rd, v = vn * rd;
                const float w = col.weight(c, ivz, scale, Z, u, v, ok);
                if (!ok) continue;
                acc[k] += bilinear_view(p, nu, nv, u, v) * w;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < ZR; ++k) {
        if (z0 + k >= g.nz) break;
        const size_t at = ((size_t)(z0 + k) * g.ny + y) * g.nx + x;
        if (st.mode == OpBpStore::kUpdate) {
            float v = st.x[at] + st.lambda * acc[k] / (st.col[at] + st.eps);
            if (st.use_min && v < st.lo) v = st.lo;
            if (st.use_max && v > st.hi) v = st.hi;
            st.x[at] = v;
        } else if (st.mode == OpBpStore::kWeight) {
            volume[at] = acc[k] <= 0.f ? 1e30f : acc[k];
        } else {
            volume[at] = st.mode == OpBpStore::kAdd ? volume[at] + acc[k] : acc[k];
        }
    }
}

// Paired guarded copy of `count` views: entry (row r, column c) holds pixels
// (r, c) and (r + 1, c), for rows and columns from -kViewGuard up to the last
// guard column and the last guard row but one, zero outside the detector.
__global__ void __launch_bounds__(256)
pair_views_kernel(const float* __restrict__ proj, float2* __restrict__ out, int nu, int nv)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    const int pitch = paired_pitch(nu);
    if (e >= pitch) return;
    const int c = e - kViewGuard, r = int(blockIdx.y) - kViewGuard;
    const float* p = proj + size_t(blockIdx.z) * nu * nv;
    const bool in = c >= 0 && c < nu;
    const float a = in && r >= 0 && r < nv ? p[size_t(r) * nu + c] : 0.f;
    const float b = in && r + 1 >= 0 && r + 1 < nv ? p[size_t(r + 1) * nu + c] : 0.f;
    out[(size_t(blockIdx.z) * gridDim.y + blockIdx.y) * pitch + e] = make_float2(a, b);
}

}  // namespace

void launch_joseph_fp(const JosephLaunch& p, hipStream_t s)
{
    dim3 block(64, 4), grid((p.nu + 63) / 64, (p.nv + 3) / 4, p.count);
    hipLaunchKernelGGL(joseph_fp_kernel, grid, block, 0, s, p.volume, p.volume_t, p.proj, p.views,
        p.vol, p.nu, p.nv, p.accumulate);
    YK_HIP(hipGetLastError());
}

size_t joseph_column_size(int nx, int ny, int nz, bool x_main)
{
    const size_t g = 2 * kJosephGuard;
    return size_t(x_main ? nx : ny) * ((x_main ? ny : nx) + g) * column_pitch(nz);
}

void launch_joseph_column_copy(const float* in, float* out, int nx, int ny, int nz, bool x_main, hipStream_t s)
{
    const int g = 2 * kJosephGuard;
    dim3 block(32, 8);
    if (x_main)
        hipLaunchKernelGGL(zfast_copy_kernel<true>, dim3((nx + 31) / 32, (column_pitch(nz) + 31) / 32, ny + g), block, 0, s, in, out,
            nx, ny, nz);
    else
        hipLaunchKernelGGL(zfast_copy_kernel<false>, dim3((nx + g + 31) / 32, (column_pitch(nz) + 31) / 32, ny), block, 0, s, in, out,
            nx, ny, nz);
    YK_HIP(hipGetLastError());
}

namespace {

// Columns from which a column's slices are split over four waves instead of
// eight (each wave forms tables for its parts): 12 views of 256 x 192 at 128^3
// (3072 columns) 78.6 -> 71.8 us, 30 of 128 x 96 at 64^3 (3840) 56.5 -> 49.5; one
// view (256 and 128 columns) 31.9 -> 35.9 and 23.6 -> 25.4.
constexpr size_t kFewColumns = 2048;

// Whole columns up to which a workgroup takes four views' instead of eight: fewer
// of them end half empty, but fewer share tap rows.  Eight and four: 256^3 from 60
// views of 512 x 384 (30720 columns) 1023 and 982 us, from 360 (184320) 5.77 and 5.73
// ms; 512^3 of 1024 x 768 from 90 (92160) 16.7 and 15.6, from 720 (737280) 102.6 and
// 107.1.
constexpr size_t kFewRounds = 262144;

template <int K, bool SPLIT>
void launch_column_kernel(const JosephSepFpLaunch& p, hipStream_t s)
{
    const size_t column = size_t(column_pitch(p.vol.nz)) * sizeof(float);
    // the waves' columns in 32 KiB; a longer column has a workgroup to itself
    int waves = column <= 4096 ? kColumnWaves : column <= 8192 ? 4 : column <= 16384 ? 2 : 1;
    const size_t columns = size_t(p.nu) * p.count;
    if (SPLIT ? columns >= kFewColumns : columns <= kFewRounds) waves = std::min(waves, 4);
    const size_t lds = column * waves + (SPLIT ? size_t(kColumnParts) * 64 * K * sizeof(float) : 0);
    if (waves == 1)
        YK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(joseph_fp_column_kernel<K, SPLIT>),
            hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    dim3 grid((p.nu + 7) / 8 * 8, (p.nv + 64 * K - 1) / (64 * K), SPLIT ? p.count : (p.count + waves - 1) / waves);
    hipLaunchKernelGGL((joseph_fp_column_kernel<K, SPLIT>), grid, dim3(64 * waves), lds, s, p.vol_zx, p.vol_zy,
        p.proj, p.views, p.vol, p.nu, p.nv, p.count, p.store);
}

// A call of fewer columns than kSplitColumns (4 waves for each of 1024 SIMDs)
// takes SPLIT, and one of kRoundColumns (the waves resident at six a SIMD) to
// twice as many: a wave a column would leave the second round partly empty, and
// four a column leave shorter ones.  Whole calls, not split and split: 256^3 of
// 512 x 384, 1 view 163 and 65 us, 4 views 172 and 125; 128^3 of 128 x 96, 40
// views (5120 columns) 74 and 77, 60 views (7680) 117 and 97, 120 views (15360)
// 171 and 169; 192^3 of 192 x 144, 60 views (11520) 250 and 219.
constexpr size_t kSplitColumns = 4096, kRoundColumns = 6144;

template <int K>
void launch_column(const JosephSepFpLaunch& p, hipStream_t s)
{
    const size_t columns = size_t(p.nu) * p.count * ((p.nv + 64 * K - 1) / (64 * K));
    const bool split = columns < kSplitColumns || (columns > kRoundColumns && columns <= 2 * kRoundColumns);
    if (split && p.count <= 65535) launch_column_kernel<K, true>(p, s);
    else launch_column_kernel<K, false>(p, s);
}

}  // namespace

bool joseph_column_fits(const VolumeGeom& g)
{
    const size_t g2 = 2 * kJosephGuard;
    const size_t slice = (size_t(std::max(g.nx, g.ny)) + g2) * size_t(column_pitch(g.nz)) * sizeof(float);
    // 128 KB of LDS for the longest column beside the tables and parts, 32-bit byte
    // offsets in a slice
    return g.nz <= 32767 && slice < (size_t(1) << 32);
}

void launch_joseph_fp_column(const JosephSepFpLaunch& p, hipStream_t s)
{
    // rays a lane: the detector's rows in equal blocks of at most 384
    const int lanes = (p.nv + 63) / 64, blocks = (lanes + 5) / 6;
    switch ((lanes + blocks - 1) / blocks) {
    case 1: launch_column<1>(p, s); break;
    case 2: launch_column<2>(p, s); break;
    case 3: launch_column<3>(p, s); break;
    case 4: launch_column<4>(p, s); break;
    case 5: launch_column<5>(p, s); break;
    default: launch_column<6>(p, s); break;
    }
    YK_HIP(hipGetLastError());
}

size_t joseph_pair_size(int nx, int ny, int nz, bool x_main)
{
    const size_t n0 = size_t(x_main ? nx : ny), n1 = size_t(x_main ? ny : nx);
    const size_t g = 2 * kJosephGuard;
    // rows x columns of float2 per slice: (nz + 2g - 1) x (n1 + 2g)
    return n0 * (size_t(nz) + g - 1) * (n1 + g) * 2;
}

void launch_joseph_pair_copy(const float* in, float* out, int nx, int ny, int nz, bool x_main, hipStream_t s, int* flag)
{
    float2* o = reinterpret_cast<float2*>(out);
    const int g = 2 * kJosephGuard;
    if (x_main) {
        dim3 block(32, 8), grid((nx + 31) / 32, (ny + g + 31) / 32, nz + g - 1);
        hipLaunchKernelGGL(pair_slab_x_kernel, grid, block, 0, s, in, o, nx, ny, nz, flag);
    } else {
        dim3 block(256), grid((nx + 255) / 256, ny, nz + g - 1);
        hipLaunchKernelGGL(pair_slab_y_kernel, grid, block, 0, s, in, o, nx, ny, nz, flag);
    }
    YK_HIP(hipGetLastError());
}

void launch_joseph_fp_slab(const JosephSepFpLaunch& p, hipStream_t s)
{
    dim3 block(64, 8), grid((p.nu + 63) / 64, p.nv, (p.count + 7) / 8);
    hipLaunchKernelGGL(joseph_fp_slab_kernel, grid, block, 0, s, p.vol_zx, p.vol_zy, p.proj, p.views, p.vol,
        p.nu, p.nv, p.count, p.store);
    YK_HIP(hipGetLastError());
}

void launch_transpose_xy(const float* in, float* out, int nx, int ny, int nz, hipStream_t s)
{
    dim3 block(32, 8), grid((nx + 31) / 32, (ny + 31) / 32, nz);
    hipLaunchKernelGGL(transpose_xy_kernel, grid, block, 0, s, in, out, nx, ny);
    YK_HIP(hipGetLastError());
}

void launch_joseph_adjoint(const JosephAdjointLaunch& p, hipStream_t s)
{
    dim3 tb(64, 4), tg((p.nu + 63) / 64, (p.nv + 3) / 4, p.count);
    hipLaunchKernelGGL(joseph_ray_table_kernel, tg, tb, 0, s, p.views, p.vol, p.nu, p.nv, p.ray_ab, p.ray_len);
    dim3 block(256), grid((p.vol.nx + 15) / 16, (p.vol.ny + 15) / 16, p.vol.nz);
    hipLaunchKernelGGL(joseph_adjoint_kernel, grid, block, 0, s, p.proj, p.volume, p.views, p.coeff32,
        p.ray_ab, p.ray_len, p.vol, p.nu, p.nv, p.count, p.accumulate);
    YK_HIP(hipGetLastError());
}

void launch_joseph_ones(const JosephLaunch& p, hipStream_t s)
{
    dim3 block(64, 4), grid((p.nu + 63) / 64, (p.nv + 3) / 4, p.count);
    hipLaunchKernelGGL(joseph_ones_kernel, grid, block, 0, s, p.proj, p.views, p.vol, p.nu, p.nv);
    YK_HIP(hipGetLastError());
}

void launch_siddon_ones(const SiddonLaunch& p, hipStream_t s)
{
    dim3 block(64, 4), grid((p.nu + 63) / 64, (p.nv + 3) / 4, p.count);
    hipLaunchKernelGGL(siddon_ones_kernel, grid, block, 0, s, p.proj, p.views, p.vol, p.nu, p.nv);
    YK_HIP(hipGetLastError());
}

void launch_siddon_fp(const SiddonLaunch& p, hipStream_t s)
{
    dim3 block(256), grid((p.nu + 7) / 8, (p.nv + 3) / 4, (p.count + 7) / 8);
    hipLaunchKernelGGL(siddon_fp_kernel, grid, block, 0, s, p.volume, p.proj, p.views, p.vol, p.nu,
        p.nv, p.count, p.accumulate);
    YK_HIP(hipGetLastError());
}

void launch_clear_flag(int* flag, hipStream_t s)
{
    hipLaunchKernelGGL(clear_flag_kernel, dim3(1), dim3(1), 0, s, flag);
    YK_HIP(hipGetLastError());
}

void launch_siddon_fp_slab(const SiddonSlabFpLaunch& p, hipStream_t s)
{
    dim3 block(64, 8), grid((p.nu + 63) / 64, p.nv, (p.count + 7) / 8);
    hipLaunchKernelGGL(siddon_fp_slab_kernel, grid, block, 0, s, p.vol_x, p.vol_y, p.volume, p.flag, p.proj, p.views,
        p.vol, p.nu, p.nv, p.count, p.accumulate);
    YK_HIP(hipGetLastError());
}

void launch_siddon_adjoint(const SiddonAdjointLaunch& p, hipStream_t s)
{
    dim3 block(256), grid((p.vol.nx + 15) / 16, (p.vol.ny + 15) / 16, p.vol.nz);
    hipLaunchKernelGGL(siddon_adjoint_kernel, grid, block, 0, s, p.proj, p.volume, p.views, p.coeff32,
        p.vol, p.nu, p.nv, p.count, p.accumulate);
    YK_HIP(hipGetLastError());
}

size_t paired_view_floats(int nu, int nv) { return size_t(paired_rows(nv)) * paired_pitch(nu) * 2; }

namespace {

// Workgroups of kOpBpZ slices from which a launch takes them; below, a lane runs
// 2 slices in four times the workgroups, else the GPU is not filled.  Whole
// calls of voxel-driven Joseph, 8 and 2 slices: 60 views at 32^3 116 and 52 us,
// 64^3 120 and 58, 96^3 137 and 107, 128^3 (1024 workgroups) 199 and 202, 160^3
// 311 and 347; one view at 64^3 19.0 and 16.4, at 256^3 43 and 48.
constexpr long kOpWideBlocks = 1024;

template <int MODE, int ZR>
void launch_op_run(const OpBpLaunch& p, hipStream_t s)
{
    const int z_blocks = (p.vol.nz + ZR - 1) / ZR;
    dim3 block(256), grid((p.vol.nx + 15) / 16, (p.vol.ny + 15) / 16, z_blocks * (p.units ? p.n_units : 1));
    auto k = !p.paired ? fdk_operator_bp_kernel<MODE, false, false, ZR>
        : p.front      ? fdk_operator_bp_kernel<MODE, true, true, ZR>
                       : fdk_operator_bp_kernel<MODE, true, false, ZR>;
    hipLaunchKernelGGL(k, grid, block, 0, s, p.paired ? p.paired : p.proj, p.volume, p.views, p.vol, p.nu, p.nv, p.count,
        p.scale, p.one_view ? 0 : 1, p.units, z_blocks, p.store);
}

template <int MODE>
void launch_op(const OpBpLaunch& p, hipStream_t s)
{
    const long wide = long((p.vol.nx + 15) / 16) * ((p.vol.ny + 15) / 16) * ((p.vol.nz + kOpBpZ - 1) / kOpBpZ) *
        (p.units ? p.n_units : 1);
    if (wide >= kOpWideBlocks) launch_op_run<MODE, kOpBpZ>(p, s);
    else launch_op_run<MODE, kOpBpShortZ>(p, s);
}

}  // namespace

void launch_fdk_operator_bp(const OpBpLaunch& p, hipStream_t s)
{
    if (p.paired) {
        dim3 grid((paired_pitch(p.nu) + 255) / 256, paired_rows(p.nv), p.one_view ? 1 : p.count);
        hipLaunchKernelGGL(pair_views_kernel, grid, dim3(256), 0, s, p.proj, reinterpret_cast<float2*>(p.paired), p.nu, p.nv);
    }
    if (p.mode == kOpMatched) launch_op<kOpMatched>(p, s);
    else if (p.mode == kOpJosephVoxel) launch_op<kOpJosephVoxel>(p, s);
    else launch_op<kOpFdk>(p, s);
    YK_HIP(hipGetLastError());
}

}  // namespace yk
