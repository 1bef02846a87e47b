// Projection-operator plan: per-view device records for the Joseph and
// Siddon forward models and their transposes, and the iterative callers
// (CGLS, SART) built on them.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "fdk.hpp"

using namespace yk;

namespace {

// Samples (voxels x views) or views from which the operator-form
// backprojections sample a paired copy of the views, and the voxels per pixel
// below which the copy is most of the work: one view at 64^3 takes 8.7 us with
// the copy and 6.4 without, two 8.5 and 9.1, four 10.0 and 15.4; one view at
// 128^3 8.8 and 10.0, at 256^3 29 and 43; four views at 32^3 9.9 and 14.6.
constexpr double kOpPairSamples = 1e6, kOpPairRatio = 0.5;
constexpr int kOpPairViews = 3;

// rays x main-axis slabs of all the plan's views per voxel from which the Siddon
// projection makes its volume copies.  Calls of a plan of 60 views, walk and
// copies with the slab kernel: at 128^3 one view of 128 x 96 59 and 34 us, all 301
// and 114; at 256^3 one view of 256 x 192 145 and 120 us, all 3370 and 836, of
// 64 x 48 136 and 116, 361 and 367; at 512^3 one view of 512 x 384 0.79 and 0.87
// ms, all 32.7 and 8.3.  Few views of a coarse detector before a large volume lose
// by it (512^3, one view of 256 x 192: 0.39 and 0.72 ms): the walk reads only what
// their rays cross, but a ray must not depend on the call it is in.
constexpr double kSiddonSlabRatio = 1.0;

// Samples (voxels x views) from which the Joseph transpose of separable views goes
// by columns; it takes three launches and passes over two volumes more than the
// gather, so a single view never does.  Gather and columns, detector as wide as
// the volume: 96^3 x 4 views 16 and 21 us, x 8 26 and 26, x 60 136 and 95; 128^3
// x 1 12 and 19, x 4 28 and 26, x 60 251 and 126; 256^3 x 1 39 and 51, x 2 66 and
// 58, x 60 1535 and 500; 64^3 x 30 37 and 39, x 60 63 and 61.
constexpr double kColumnSamples = 8e6;
constexpr int kColumnViews = 2;

// Rays up to which a Joseph projection's store makes the solvers' residual: its
// lanes run along detector columns, so the reads of b and the row weights it
// adds are scattered.  One view of 128 x 96 saves 2.5 us by it, 12 views of 256 x
// 192 (590 000 rays) lose 1 us.
constexpr size_t kResidualRays = 200000;

bool operator_form(int kind)
{
    return kind == YK_BP_FDK || kind == YK_BP_FDK_PSEUDO_MATCHED || kind == YK_BP_JOSEPH_VOXEL;
}

int op_mode(int kind) { return kind == YK_BP_FDK_PSEUDO_MATCHED ? 1 : kind == YK_BP_JOSEPH_VOXEL ? 2 : 0; }

// record of the gather transposes of a view whose main axis is X or Y, from
// its vectors in volume-centred voxel units and the projective map of world
// points.  In FP64: the forward kernel's float records of a source 1500 voxels
// away put a ray 4e-5 voxels aside.
void gather_view(const ViewD& w, int axis, int nu, int nv, const double map[12], const VolumeGeom& g, GatherViewDev& o)
{
    std::memset(&o, 0, sizeof(o));
    o.axis = axis;
    const int order[3] = { axis, axis == 0 ? 1 : 0, 2 };
    double most = 0.0;
    for (int a = 0; a < 4; ++a)
        most = std::max(most, std::fabs(w.detS[axis] - w.src[axis] + ((a & 1) ? nu - 1 : 0) * w.detU[axis] +
            ((a & 2) ? nv - 1 : 0) * w.detV[axis]));
    int e = 0;
    std::frexp(most, &e);
    const double scale = std::ldexp(1.0, -e);
    o.scale = float(scale);
    double* rows[3] = { o.d, o.e1, o.e2 };
    for (int k = 0; k < 3; ++k) {
        const int c = order[k];
        o.src[k] = w.src[c];
        rows[k][0] = (w.detS[c] - w.src[c]) * scale;
        rows[k][1] = w.detU[c] * scale;
        rows[k][2] = w.detV[c] * scale;
    }
    // the map at voxel index (i, j, k): X = origin + index x voxel
    const double vox[3] = { g.vx, g.vy, g.vz }, org[3] = { g.ox, g.oy, g.oz };
    float* maps[3] = { o.mu, o.mv, o.md };
    for (int m = 0; m < 3; ++m) {
        const double* c = map + 4 * m;
        for (int k = 0; k < 3; ++k) maps[m][k] = float(c[k] * vox[k]);
        maps[m][3] = float(c[0] * org[0] + c[1] * org[1] + c[2] * org[2] + c[3]);
    }
}

// Which of X (1) and Y (2) may be the main axis, the larger |ray / voxel|, of some
// ray of the view.  The ray is linear over the detector, so where one component
// keeps its sign and exceeds the other's size at the corners it does everywhere.
int ray_axes(const ViewD& w, const double vox[3], int nu, int nv)
{
    bool x_only = true, y_only = true;
    double sign[2] = { 0.0, 0.0 };
    for (int a = 0; a < 4; ++a) {
        double r[2];
        for (int k = 0; k < 2; ++k) {
            r[k] = (w.detS[k] + ((a & 1) ? nu - 1 : 0) * w.detU[k] + ((a & 2) ? nv - 1 : 0) * w.detV[k] - w.src[k]) / vox[k];
            if (sign[k] == 0.0) sign[k] = r[k] < 0.0 ? -1.0 : 1.0;
        }
        // (a margin for the kernel's own rounding)
        x_only = x_only && sign[0] * r[0] > 1.000001 * std::fabs(r[1]);
        y_only = y_only && sign[1] * r[1] > 1.000001 * std::fabs(r[0]);
    }
    return x_only ? 1 : y_only ? 2 : 3;
}

// The plane between cells (0 .. n) on which the source lies along an axis, or
// -1.  The tolerance is twice the rounding that the voxels' FP32 origin and size
// bring to a plane: a centred scan has its source in the middle plane of an even
// volume, whatever the voxel.
int source_plane(double src, double centre, double voxel, int n)
{
    const double cell = (src - centre) / voxel + 0.5 * n, plane = std::rint(cell);
    return plane >= 0.0 && plane <= n && std::fabs(cell - plane) <= n * 0x1p-23 ? int(plane) : -1;
}

// No ray of the view runs across its main axis: the general Siddon gather
// measures segments along that axis
bool along_main(const ViewD& w, int axis, int nu, int nv)
{
    double sign = 0.0;
    for (int a = 0; a < 4; ++a) {
        double r[3], len2 = 0.0;
        for (int k = 0; k < 3; ++k) {
            r[k] = w.detS[k] + ((a & 1) ? nu - 1 : 0) * w.detU[k] + ((a & 2) ? nv - 1 : 0) * w.detV[k] - w.src[k];
            len2 += r[k] * r[k];
        }
        // (linear over the detector: its corners bound it)
        if (sign == 0.0) sign = r[axis] < 0.0 ? -1.0 : 1.0;
        if (!(sign * r[axis] > 1e-3 * std::sqrt(len2))) return false;
    }
    return true;
}

// The column transpose takes separable views in which at most eight rays of a
// detector column pass within a voxel along z, of a detector whose row
// numbers times FP32 rounding stay far below its 0.01 pixels of margin
bool column_view(const ProjViewDev& p, int nu, int nv, const VolumeGeom& g)
{
    const int a = p.axis;
    const double h = 0.5 * ((a == 0 ? g.nx : g.ny) - 1);
    const double near = std::fabs(double(p.src[a])) - h;  // least distance of a slice from the source
    double far = 0.0;
    for (int u : { 0, nu - 1 }) far = std::max(far, std::fabs(double(p.detS[a]) + u * double(p.detU[a]) - p.src[a]));
    return near > 0.0 && nv <= 8192 && far <= 3.9 * near * std::fabs(double(p.detV[2]));
}

// least and largest distance of the volume's voxels, grown by `xy` and `z`
// voxels on each side, from the source plane (row 2 of the map), over the
// detector plane's
void depth_range(const yk_view& w, const double map[12], const VolumeGeom& g, double xy, double z, double& least,
    double& most)
{
    const ViewD d = widen(w);
    const double plane = map[8] * d.detS[0] + map[9] * d.detS[1] + map[10] * d.detS[2] + map[11];
    least = 1e300;
    most = -1e300;
    for (int a = 0; a < 8; ++a) {
        const double X = g.ox + ((a & 1) ? g.nx - 1 + xy : -xy) * double(g.vx);
        const double Y = g.oy + ((a & 2) ? g.ny - 1 + xy : -xy) * double(g.vy);
        const double Z = g.oz + ((a & 4) ? g.nz - 1 + z : -z) * double(g.vz);
        const double depth = (map[8] * X + map[9] * Y + map[10] * Z + map[11]) / plane;
        least = std::min(least, depth);
        most = std::max(most, depth);
    }
}

}  // namespace

yk_projector::yk_projector(yk_ctx* c, const yk_view* v, int n, int nu_, int nv_,
    const yk_volume_grid& g, float range, const std::vector<int>* segments)
    : ctx(c), nu(nu_), nv(nv_), n_views(n), grid(g),
      scan_range(range > 0.f ? double(range) : 6.28318530717958647692)
{
    if (!v || n <= 0) fail(YK_ERR_INVALID_GEOMETRY, "projector needs at least one view");
    if (nu <= 0 || nv <= 0) fail(YK_ERR_INVALID_GEOMETRY, "invalid detector size");
    validate_volume(grid);
    views.assign(v, v + n);
    vol = volume_geom(grid);
    ctx->activate();
    std::vector<ProjViewDev> jv(n);
    std::vector<SiddonViewDev> sv(n);
    std::vector<double> c64(size_t(n) * 12);
    std::vector<GatherViewDev> gv(n);
    const double vox[3] = { grid.voxel_x_mm, grid.voxel_y_mm, grid.voxel_z_mm };
    const double cen[3] = { grid.center_mm[0], grid.center_mm[1], grid.center_mm[2] };
    for (int i = 0; i < n; ++i) {
        const yk_view& w = views[i];
        for (int k = 0; k < 3; ++k)
            if (!std::isfinite(w.src[k]) || !std::isfinite(w.detS[k]) || !std::isfinite(w.detU[k]) ||
                !std::isfinite(w.detV[k]))
                fail(YK_ERR_INVALID_GEOMETRY, "non-finite view vector");
        // normalizeToVoxel (src/common/cuda/operators/YkOperatorKernelTypes.cuh:148-168)
        ProjViewDev& p = jv[i];
        std::memset(&p, 0, sizeof(p));
        for (int k = 0; k < 3; ++k) {
            p.src[k] = float((double(w.src[k]) - cen[k]) / vox[k]);
            p.detS[k] = float((double(w.detS[k]) - cen[k]) / vox[k]);
            p.detU[k] = float(double(w.detU[k]) / vox[k]);
            p.detV[k] = float(double(w.detV[k]) / vox[k]);
        }
        p.axis = main_axis(w, nu, nv);
        if (p.axis == 0) any_x_axis = true;
        // d0 and d1 of every ray independent of v (exact zeros, so bit-exact)
        separable.push_back(p.axis != 2 && p.detV[p.axis == 0 ? 0 : 1] == 0.f &&
                            p.detV[p.axis == 0 ? 1 : 0] == 0.f);
        SiddonViewDev& s = sv[i];
        std::memset(&s, 0, sizeof(s));
        std::memcpy(s.src, w.src, sizeof(s.src));
        std::memcpy(s.detS, w.detS, sizeof(s.detS));
        std::memcpy(s.detU, w.detU, sizeof(s.detU));
        std::memcpy(s.detV, w.detV, sizeof(s.detV));
        siddon_axes.push_back(char(ray_axes(widen(w), vox, nu, nv)));
        const int cells[3] = { grid.nx, grid.ny, grid.nz };
        const float lo[3] = { vol.ox - 0.5f * vol.vx, vol.oy - 0.5f * vol.vy, vol.oz - 0.5f * vol.vz };
        for (int k = 0; k < 3; ++k) {
            s.plane[k] = source_plane(w.src[k], cen[k], vox[k], cells[k]);
            s.on_plane[k] = s.plane[k] < 0 ? w.src[k] : std::fma(float(s.plane[k]), float(vox[k]), lo[k]);
        }
        projection_map(w, &c64[size_t(i) * 12]);
        // Gather transposes.  Their kernels take every support of a run of
        // kGatherRun voxels to lie before the source, and the general Siddon one
        // that the detector ends no ray inside the volume.
        if (p.axis != 2) {
            const double* map = &c64[size_t(i) * 12];
            double least, most, inner, outer;
            depth_range(w, map, vol, 2.0, kGatherRun + 2.0, least, most);
            depth_range(w, map, vol, 0.5, 0.5, inner, outer);
            ViewD n{};
            for (int k = 0; k < 3; ++k) {
                n.src[k] = (double(w.src[k]) - cen[k]) / vox[k];
                n.detS[k] = (double(w.detS[k]) - cen[k]) / vox[k];
                n.detU[k] = double(w.detU[k]) / vox[k];
                n.detV[k] = double(w.detV[k]) / vox[k];
            }
            gather_view(n, p.axis, nu, nv, map, vol, gv[i]);
            const bool front = least > 1e-3;
            near_source.push_back(!front);
            joseph_gather.push_back(front);
            siddon_gather.push_back(front && outer < 1.0 && along_main(widen(w), p.axis, nu, nv));
            siddon_flat.push_back(front && separable.back() && w.detU[2] == 0.f);
            siddon_ends.push_back(!(outer < 1.0));
            joseph_column.push_back(front && separable.back() && column_view(p, nu, nv, vol));
        } else {
            near_source.push_back(0);
            joseph_gather.push_back(0);
            siddon_gather.push_back(0);
            joseph_column.push_back(0);
            siddon_flat.push_back(0);
            siddon_ends.push_back(0);
        }
    }
    d_gather.upload(gv.data(), gv.size(), ctx->stream);
    // operator-form FDK backprojection records (FP64 geometry over the whole
    // view sequence, like FdkAffineCoeff in .../FDK/kernels/YkFDKBpPrecompute.cu:14-138)
    std::vector<DerivedD> der;
    std::vector<CoeffD> cf;
    if (segments) {
        std::vector<DerivedD> sder;
        std::vector<CoeffD> scf;
        auto at = views.begin();
        for (int k : *segments) {
            const std::vector<yk_view> part(at, at + k);
            derive_geometry(part, nu, nv, scan_range, sder);
            fdk_coefficients(part, sder, scf);
            der.insert(der.end(), sder.begin(), sder.end());
            cf.insert(cf.end(), scf.begin(), scf.end());
            at += k;
        }
    } else {
        derive_geometry(views, nu, nv, scan_range, der);
        fdk_coefficients(views, der, cf);
    }
    std::vector<OpBpViewDev> ov(n);
    op_scale.resize(n);
    for (int i = 0; i < n; ++i) {
        const ViewD w = widen(views[i]);
        OpBpViewDev& o = ov[i];
        std::memset(&o, 0, sizeof(o));
        for (int k = 0; k < 4; ++k) {
            o.cu[k] = float(cf[i].cu[k]);
            o.cv[k] = float(cf[i].cv[k]);
            o.cd[k] = float(cf[i].cd[k]);
        }
        const double sod = der[i].sod;
        for (int k = 0; k < 3; ++k) {
            o.cc[k] = float(-w.src[k] / sod);
            o.src[k] = float(w.src[k]);
        }
        o.cc[3] = float(sod);
        double r0[3];
        for (int k = 0; k < 3; ++k) r0[k] = w.detS[k] - w.src[k];
        auto dot = [](const double* a, const double* b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; };
        o.l2[0] = float(dot(r0, r0));
        o.l2[1] = float(2.0 * dot(r0, w.detU));
        o.l2[2] = float(2.0 * dot(r0, w.detV));
        o.l2[3] = float(dot(w.detU, w.detU));
        o.l2[4] = float(2.0 * dot(w.detU, w.detV));
        o.l2[5] = float(dot(w.detV, w.detV));
        o.wbase = float(cf[i].wbase);
        o.inv_sdd_plane = std::fabs(der[i].sdd_plane) > 1e-12 ? float(1.0 / std::fabs(der[i].sdd_plane)) : 0.f;
        // depth and FDK weight denominator (both affine) over the voxels and
        // a run's overhang past the last slice
        double least = 1e300;
        for (int a = 0; a < 8; ++a) {
            const double X = vol.ox + ((a & 1) ? (vol.nx - 1) * double(vol.vx) : 0.0);
            const double Y = vol.oy + ((a & 2) ? (vol.ny - 1) * double(vol.vy) : 0.0);
            const double Z = vol.oz + ((a & 4) ? (vol.nz + 7) * double(vol.vz) : 0.0);
            const double* d = cf[i].cd;
            least = std::min({ least, (d[0] * X + d[1] * Y + d[2] * Z + d[3]) / der[i].sdd_plane,
                               1.0 - (w.src[0] * X + w.src[1] * Y + w.src[2] * Z) / (sod * sod) });
        }
        op_front.push_back(least > 1e-3);
        op_scale[i] = vox[0] * vox[1] * vox[2] / der[i].du / der[i].dv;
    }
    hipStream_t s = ctx->stream;
    d_opviews.upload(ov.data(), ov.size(), s);
    d_jviews.upload(jv.data(), jv.size(), s);
    d_sviews.upload(sv.data(), sv.size(), s);
    std::vector<float> c32(c64.begin(), c64.end());
    d_c32.upload(c32.data(), c32.size(), s);
    d_partials.resize(1024);
    YK_HIP(hipStreamSynchronize(s));
}

void yk_projector::note_capture()
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &status) != hipSuccess) {
        (void)hipGetLastError();  // (the null stream beside another's capture: the launches say what is wrong)
        status = hipStreamCaptureStatusNone;
    }
    capturing = status != hipStreamCaptureStatusNone;
    captured = captured || capturing;
}

float* SolverScratch::array(int k, size_t n)
{
    if (arrays[k].size() < n) arrays[k].resize(n);
    return arrays[k].get();
}

SolverScratch::~SolverScratch() = default;

SolverCall::~SolverCall()
{
    (void)hipStreamSynchronize(stream);
    size_t bytes = 0;
    for (const auto& a : ws.arrays) bytes += a.size() * sizeof(float);
    if (bytes > SolverScratch::kKeep)
        for (auto& a : ws.arrays) a.reset();
    ws.busy = false;
}

// the paired slab copies of the volume for rays of either main axis into w's
// scratch; false when the walk, which needs none, has to serve the call: the
// copies do not fit in memory, a stream capture allows no allocation, or the slab
// kernel's grid or 32-bit slab offsets cannot hold the sizes
bool yk_projector::siddon_copies(yk_projector& w, const float* d_volume, bool any_x, bool any_y)
{
    const size_t size_x = joseph_pair_size(grid.nx, grid.ny, grid.nz, true);
    const size_t size_y = joseph_pair_size(grid.nx, grid.ny, grid.nz, false);
    if (nv > 65535 || size_x / grid.nx > (size_t(1) << 29) || size_y / grid.ny > (size_t(1) << 29)) return false;
    const size_t need_x = any_x ? size_x : 0, need_y = any_y ? size_y : 0;
    if (w.d_vol_zx.size() < need_x || w.d_vol_zy.size() < need_y || !w.d_flag.get()) {
        if (w.capturing) return false;
    }
    try {
        w.grow(w.d_vol_zx, need_x);
        w.grow(w.d_vol_zy, need_y);
        w.grow(w.d_flag, 1);
    } catch (const Error&) {
        (void)hipGetLastError();  // the failed allocation's, not the call's
        return false;
    }
    int* const flag = w.d_flag.get();
    launch_clear_flag(flag, ctx->stream);
    if (any_x) launch_joseph_pair_copy(d_volume, w.d_vol_zx.get(), grid.nx, grid.ny, grid.nz, true, ctx->stream, flag);
    if (any_y) launch_joseph_pair_copy(d_volume, w.d_vol_zy.get(), grid.nx, grid.ny, grid.nz, false, ctx->stream, flag);
    return true;
}

bool yk_projector::project(int kind, const float* d_volume, float* d_proj, int first, int count,
    int accumulate, const FpStore* residual)
{
    if (first < 0 || count <= 0 || first + count > n_views) fail(YK_ERR_INVALID_CONFIG, "view range outside the plan");
    if (!d_volume || !d_proj) fail(YK_ERR_INVALID_BUFFER, "null device buffer");
    hipStream_t s = ctx->stream;
    yk_projector& w = scratch_owner ? *scratch_owner : *this;  // scratch arrays
    w.note_capture();
    if (size_t(count) * nu * nv > kResidualRays) residual = nullptr;
    FpStore store{};
    store.mode = accumulate ? FpStore::kAdd : FpStore::kSet;
    if (residual) store = *residual;
    bool all_sep = true, any_x = false, any_y = false, any_z = false;
    for (int i = first; i < first + count; ++i) {
        all_sep = all_sep && separable[i];
        const int ax = main_axis(views[i], nu, nv);
        any_x = any_x || ax == 0;
        any_y = any_y || ax == 1;
        any_z = any_z || ax == 2;
    }
    if (kind == YK_FP_JOSEPH && all_sep && joseph_column_fits(vol)) {
        // guarded copies (every call rewrites the copy it reads)
        if (any_x) {
            w.grow(w.d_vol_zx, joseph_column_size(grid.nx, grid.ny, grid.nz, true));
            launch_joseph_column_copy(d_volume, w.d_vol_zx.get(), grid.nx, grid.ny, grid.nz, true, s);
        }
        if (any_y) {
            w.grow(w.d_vol_zy, joseph_column_size(grid.nx, grid.ny, grid.nz, false));
            launch_joseph_column_copy(d_volume, w.d_vol_zy.get(), grid.nx, grid.ny, grid.nz, false, s);
        }
        JosephSepFpLaunch p{};
        p.vol_zx = any_x ? w.d_vol_zx.get() : nullptr;
        p.vol_zy = any_y ? w.d_vol_zy.get() : nullptr;
        p.proj = d_proj;
        p.views = d_jviews.get() + first;
        p.vol = vol;
        p.nu = nu; p.nv = nv; p.count = count;
        p.store = store;
        launch_joseph_fp_column(p, s);
        return residual != nullptr;
    } else if (kind == YK_FP_JOSEPH && !any_z) {
        // X/Y-main views of any orientation: paired slab copies
        if (any_x) {
            w.grow(w.d_vol_zx, joseph_pair_size(grid.nx, grid.ny, grid.nz, true));
            launch_joseph_pair_copy(d_volume, w.d_vol_zx.get(), grid.nx, grid.ny, grid.nz, true, s);
        }
        if (any_y) {
            w.grow(w.d_vol_zy, joseph_pair_size(grid.nx, grid.ny, grid.nz, false));
            launch_joseph_pair_copy(d_volume, w.d_vol_zy.get(), grid.nx, grid.ny, grid.nz, false, s);
        }
        JosephSepFpLaunch p{};
        p.vol_zx = any_x ? w.d_vol_zx.get() : nullptr;
        p.vol_zy = any_y ? w.d_vol_zy.get() : nullptr;
        p.proj = d_proj;
        p.views = d_jviews.get() + first;
        p.vol = vol;
        p.nu = nu; p.nv = nv; p.count = count;
        p.store = store;
        launch_joseph_fp_slab(p, s);
        return residual != nullptr;
    } else if (kind == YK_FP_JOSEPH) {
        bool need_t = false;
        std::vector<ProjViewDev> dummy;
        for (int i = first; i < first + count; ++i)
            if (main_axis(views[i], nu, nv) == 0) need_t = true;
        if (need_t) {
            w.grow(w.d_vol_t, size_t(grid.nx) * grid.ny * grid.nz);
            launch_transpose_xy(d_volume, w.d_vol_t.get(), grid.nx, grid.ny, grid.nz, s);
        }
        JosephLaunch p{};
        p.volume = d_volume;
        p.volume_t = need_t ? w.d_vol_t.get() : nullptr;
        p.proj = d_proj;
        p.views = d_jviews.get() + first;
        p.vol = vol;
        p.nu = nu; p.nv = nv; p.count = count;
        p.accumulate = accumulate;
        launch_joseph_fp(p, s);
    } else if (kind == YK_FP_SIDDON) {
        // The slab kernel reads paired copies of the volume, made on each call.
        // Which form takes a ray is the plan's matter, not the call's: the two
        // differ in rounding, and a range of views has the bits of the whole.
        const double slabs = double(n_views) * nu * nv * std::max(grid.nx, grid.ny);
        int axes = 0;
        for (int i = first; i < first + count; ++i) axes |= siddon_axes[i];
        if (slabs >= kSiddonSlabRatio * double(grid.nx) * grid.ny * grid.nz &&
            siddon_copies(w, d_volume, (axes & 1) != 0, (axes & 2) != 0)) {
            SiddonSlabFpLaunch p{};
            p.volume = d_volume;
            p.vol_x = (axes & 1) ? w.d_vol_zx.get() : nullptr;
            p.vol_y = (axes & 2) ? w.d_vol_zy.get() : nullptr;
            p.flag = w.d_flag.get();
            p.proj = d_proj;
            p.views = d_sviews.get() + first;
            p.vol = vol;
            p.nu = nu; p.nv = nv; p.count = count;
            p.accumulate = accumulate;
            launch_siddon_fp_slab(p, s);
            return false;
        }
        SiddonLaunch p{};
        p.volume = d_volume;
        p.proj = d_proj;
        p.views = d_sviews.get() + first;
        p.vol = vol;
        p.nu = nu; p.nv = nv; p.count = count;
        p.accumulate = accumulate;
        launch_siddon_fp(p, s);
    } else {
        fail(YK_ERR_UNSUPPORTED, "unknown forward projector");
    }
    return false;
}

void yk_projector::project_ones(int kind, float* d_proj, int first, int count)
{
    constexpr int kViews = 32768;  // (a grid holds 65535)
    for (int at = 0; at < count; at += kViews) {
        float* proj = d_proj + size_t(nu) * nv * at;
        if (kind == YK_FP_JOSEPH) {
            JosephLaunch p{};
            p.proj = proj;
            p.views = d_jviews.get() + first + at;
            p.vol = vol;
            p.nu = nu; p.nv = nv; p.count = std::min(kViews, count - at);
            launch_joseph_ones(p, ctx->stream);
        } else {
            SiddonLaunch p{};
            p.proj = proj;
            p.views = d_sviews.get() + first + at;
            p.vol = vol;
            p.nu = nu; p.nv = nv; p.count = std::min(kViews, count - at);
            launch_siddon_ones(p, ctx->stream);
        }
    }
}

// views per paired copy of the operator-form backprojections (one_view: the
// copy holds one view, which serves all `count`); 0: sample the
// views themselves (few samples for the copy's launch and pass, sizes past its
// grid or 24-bit row products, or no memory)
int yk_projector::op_chunk(yk_projector& w, int count, bool one_view) const
{
    const size_t per_view = paired_view_floats(nu, nv);
    const double samples = double(grid.nx) * grid.ny * grid.nz * count;
    const double copied = double(nu) * nv * (one_view ? 1 : count);
    if ((samples < kOpPairSamples && count < kOpPairViews) || samples < kOpPairRatio * copied) return 0;
    if (nv > 65000 || nu > 2000000 || per_view > (size_t(1) << 29)) return 0;
    const int chunk = one_view ? 1
        : int(std::max<size_t>(1, std::min({ size_t(count), size_t(65535), (size_t(1) << 28) / per_view })));
    if (w.d_paired_views.size() < per_view * chunk) {
        if (w.capturing) return 0;
        try {
            w.grow(w.d_paired_views, per_view * chunk);
        } catch (const Error&) {
            (void)hipGetLastError();
            return 0;
        }
    }
    return chunk;
}

// Consecutive views [first, first + count) of one transpose: the form of untilted
// views, the general gather, or the search that takes any view.  A view of another
// form splits the call instead of deciding for all of it: 128^3 x 180 untilted
// views and one tilted, Joseph 1.34 -> 0.64 ms, Siddon 1.24 -> 0.88.  A run of
// fewer than kShortRun views beside general ones joins them, as every run is a pass
// over the volume.  Two kinds of views do decide for the call:
// - a voxel within the gathers' margin of the source has thousands of candidates
//   in few lanes, which launches of few views would wait for one after another
//   (92 mm orbit around that volume, tilted: the search 31 ms, split 68); untilted
//   views are scattered then (7.4 ms);
// - rays so dense that the columns take them in some views and not in others cost
//   columns and gather alike, in twice the launches (125 mm: 1.66 ms, split 3.22).
std::vector<yk_projector::TransposeRun> yk_projector::transpose_runs(bool siddon, int first, int count) const
{
    constexpr int kShortRun = 8;
    const std::vector<char>& untilted = siddon ? siddon_flat : joseph_column;
    const std::vector<char>& general = siddon ? siddon_gather : joseph_gather;
    bool columns = true, near = false, all_sep = true;
    for (int i = first; i < first + count; ++i) {
        near = near || near_source[i];
        all_sep = all_sep && separable[i];
        columns = columns && (siddon || untilted[i] || !general[i] || !separable[i]);
    }
    if (near) return { TransposeRun{ all_sep ? kScatter : kSearch, first, count } };
    std::vector<TransposeRun> runs;
    for (int i = first; i < first + count; ++i) {
        const TransposeForm form = untilted[i] && columns ? kUntilted : general[i] ? kGeneral : kSearch;
        if (runs.empty() || runs.back().form != form) runs.push_back(TransposeRun{ form, i, 0 });
        ++runs.back().count;
    }
    std::vector<TransposeRun> joined;
    for (size_t k = 0; k < runs.size(); ++k) {
        TransposeRun r = runs[k];
        const bool beside = (k > 0 && runs[k - 1].form == kGeneral) || (k + 1 < runs.size() && runs[k + 1].form == kGeneral);
        if (r.form == kUntilted && r.count < kShortRun && beside &&
            std::all_of(general.begin() + r.first, general.begin() + r.first + r.count, [](char c) { return c != 0; }))
            r.form = kGeneral;
        if (!joined.empty() && joined.back().form == r.form) joined.back().count += r.count;
        else joined.push_back(r);
    }
    return joined;
}

// Transposes by the gather kernels, a chunk of views' table at a time (at most 1
// GiB); false when they do not apply: rows past 32-bit offsets, or no memory for
// the table (none may be allocated under a stream capture)
bool yk_projector::gather_transpose(yk_projector& w, int model, const float* d_proj, float* d_volume, int first, int count,
    int accumulate)
{
    const bool flat = model == kGatherSiddonFlat || model == kGatherSiddonFlatEnds;
    const int pitch = nu + kGatherPad;
    // floats (flat: an entry a column and a row more, columns' aligned to 8 bytes)
    const size_t rows = size_t(nv) + kGatherPadRows;
    const size_t per_view = flat ? rows * pitch + 2 * size_t(pitch) + rows + 1 : rows * pitch * (model == kGatherSiddon ? 3 : 1);
    if (nv + kGatherPadRows > 65535 || per_view > (size_t(1) << 30)) return false;
    const int chunk = int(std::max<size_t>(1, std::min({ size_t(count), size_t(65535), (size_t(1) << 28) / per_view })));
    if (w.d_gather_q.size() < per_view * chunk || !w.d_flag.get()) {
        if (w.capturing) return false;
        try {
            w.grow(w.d_gather_q, per_view * chunk);
            w.grow(w.d_flag, 1);
        } catch (const Error&) {
            (void)hipGetLastError();
            return false;
        }
    }
    for (int c0 = 0; c0 < count; c0 += chunk) {
        GatherLaunch p{};
        p.proj = d_proj + size_t(nu) * nv * c0;
        p.volume = d_volume;
        p.views = d_jviews.get() + first + c0;
        p.sviews = d_sviews.get() + first + c0;
        p.gviews = d_gather.get() + first + c0;
        p.q = w.d_gather_q.get();
        p.flag = w.d_flag.get();
        p.vol = vol;
        p.nu = nu; p.nv = nv; p.pitch = pitch; p.count = std::min(chunk, count - c0);
        p.model = model;
        if (flat) {
            const size_t q_size = (rows * pitch * p.count + 1) & ~size_t(1);
            p.ru = reinterpret_cast<float2*>(p.q + q_size);
            p.rv = p.q + q_size + 2 * size_t(pitch) * p.count;
        }
        p.accumulate = c0 > 0 ? 1 : accumulate;
        launch_gather_transpose(p, ctx->stream);
    }
    return true;
}

// Joseph transpose of separable views by detector columns, a chunk of views'
// table at a time (at most 1 GiB); false when the gather has to serve them: few
// voxels or views, or no memory
bool yk_projector::column_transpose(yk_projector& w, const float* d_proj, float* d_volume, int first, int count, int accumulate)
{
    const size_t voxels = size_t(grid.nx) * grid.ny * grid.nz;
    if (double(voxels) * count < kColumnSamples || count < kColumnViews) return false;
    const int pitch = nv + 2 * kColumnPad;
    const size_t per_view = size_t(nu) * pitch;
    if (per_view > (size_t(1) << 30)) return false;
    const int chunk = int(std::max<size_t>(1, std::min({ size_t(count), size_t(65535), (size_t(1) << 28) / per_view })));
    bool any_x = false, any_y = false;
    for (int i = first; i < first + count; ++i) (main_axis(views[i], nu, nv) == 0 ? any_x : any_y) = true;
    if (w.d_gather_q.size() < per_view * chunk || !w.d_flag.get() || (any_x && w.d_column_x.size() < voxels) ||
        (any_y && w.d_column_y.size() < voxels)) {
        if (w.capturing) return false;
        try {
            w.grow(w.d_gather_q, per_view * chunk);
            w.grow(w.d_flag, 1);
            if (any_x) w.grow(w.d_column_x, voxels);
            if (any_y) w.grow(w.d_column_y, voxels);
        } catch (const Error&) {
            (void)hipGetLastError();
            return false;
        }
    }
    for (int c0 = 0; c0 < count; c0 += chunk) {
        ColumnTransposeLaunch p{};
        p.proj = d_proj + size_t(nu) * nv * c0;
        p.volume = d_volume;
        p.views = d_jviews.get() + first + c0;
        p.gviews = d_gather.get() + first + c0;
        p.q = w.d_gather_q.get();
        p.part_x = any_x ? w.d_column_x.get() : nullptr;
        p.part_y = any_y ? w.d_column_y.get() : nullptr;
        p.flag = w.d_flag.get();
        p.vol = vol;
        p.nu = nu; p.nv = nv; p.pitch = pitch; p.count = std::min(chunk, count - c0);
        p.accumulate = c0 > 0 ? 1 : accumulate;
        launch_joseph_column_transpose(p, ctx->stream);
    }
    return true;
}

// Untilted views by scattering, a chunk of views' table at a time (at most 1 GiB);
// false when there is no memory for it (none may be allocated under a capture)
bool yk_projector::scatter_transpose(yk_projector& w, bool siddon, const float* d_proj, float* d_volume, int first, int count,
    int accumulate)
{
    // floats a view: Joseph (a2, b2) and p L of every ray, (a1, b1) of every column;
    // Siddon two a ray and two a column
    const size_t rays = size_t(nu) * (nv + kScatterPad);
    const size_t per_view = (siddon ? 2 : 3) * rays + 2 * size_t(nu);
    const int chunk = int(std::max<size_t>(1, std::min({ size_t(count), size_t(65535), (size_t(1) << 28) / per_view })));
    if (w.d_scatter.size() < per_view * chunk) {
        if (w.capturing) return false;
        try {
            w.grow(w.d_scatter, per_view * chunk);
        } catch (const Error&) {
            (void)hipGetLastError();
            return false;
        }
    }
    for (int c0 = 0; c0 < count; c0 += chunk) {
        const int n = std::min(chunk, count - c0);
        float2* const columns = reinterpret_cast<float2*>(w.d_scatter.get());
        float2* const table = columns + size_t(nu) * n;
        const float* proj = d_proj + size_t(nu) * nv * c0;
        const float* map = d_c32.get() + size_t(first + c0) * 12;
        const int add = c0 > 0 ? 1 : accumulate;
        if (siddon) {
            launch_siddon_scatter(SiddonScatterLaunch{ proj, d_volume, d_sviews.get() + first + c0, map, columns, table, vol, nu, nv,
                n, add }, ctx->stream);
        } else {
            launch_joseph_scatter(JosephScatterLaunch{ proj, d_volume, d_jviews.get() + first + c0, map, columns, table,
                reinterpret_cast<float*>(table + rays * n), vol, nu, nv, n, add }, ctx->stream);
        }
    }
    return true;
}

// one run of transpose_runs
void yk_projector::transpose(yk_projector& w, bool siddon, TransposeForm form, const float* d_proj, float* d_volume, int first,
    int count, int accumulate)
{
    hipStream_t s = ctx->stream;
    const bool ends = std::any_of(siddon_ends.begin() + first, siddon_ends.begin() + first + count, [](char c) { return c != 0; });
    const int model = !siddon ? kGatherJoseph : form != kUntilted ? kGatherSiddon : ends ? kGatherSiddonFlatEnds : kGatherSiddonFlat;
    if (form == kScatter && scatter_transpose(w, siddon, d_proj, d_volume, first, count, accumulate)) return;
    if (!siddon && form == kUntilted && column_transpose(w, d_proj, d_volume, first, count, accumulate)) {
    } else if (form <= kGeneral && gather_transpose(w, model, d_proj, d_volume, first, count, accumulate)) {
    } else if (!siddon) {
        // the ray table holds a chunk of views at a time (at most 1 GiB)
        const size_t per_view = size_t(nu) * nv;
        const int chunk = int(std::max<size_t>(1, std::min<size_t>(size_t(count),
            (size_t(1) << 30) / (per_view * (sizeof(float4) + sizeof(float))))));
        w.grow(w.d_ray_ab, per_view * chunk);
        w.grow(w.d_ray_len, per_view * chunk);
        for (int c0 = 0; c0 < count; c0 += chunk) {
            JosephAdjointLaunch p{};
            p.proj = d_proj + per_view * c0;
            p.volume = d_volume;
            p.views = d_jviews.get() + first + c0;
            p.coeff32 = d_c32.get() + size_t(first + c0) * 12;
            p.ray_ab = w.d_ray_ab.get();
            p.ray_len = w.d_ray_len.get();
            p.vol = vol;
            p.nu = nu; p.nv = nv; p.count = std::min(chunk, count - c0);
            p.accumulate = c0 > 0 ? 1 : accumulate;
            launch_joseph_adjoint(p, s);
        }
    } else {
        SiddonAdjointLaunch p{};
        p.proj = d_proj;
        p.volume = d_volume;
        p.views = d_sviews.get() + first;
        p.coeff32 = d_c32.get() + size_t(first) * 12;
        p.vol = vol;
        p.nu = nu; p.nv = nv; p.count = count;
        p.accumulate = accumulate;
        launch_siddon_adjoint(p, s);
    }
}

void yk_projector::backproject(int kind, const float* d_proj, float* d_volume, int first, int count,
    int accumulate)
{
    if (first < 0 || count <= 0 || first + count > n_views) fail(YK_ERR_INVALID_CONFIG, "view range outside the plan");
    if (!d_volume || !d_proj) fail(YK_ERR_INVALID_BUFFER, "null device buffer");
    hipStream_t s = ctx->stream;
    yk_projector& w = scratch_owner ? *scratch_owner : *this;  // scratch arrays
    w.note_capture();
    if (kind == YK_BP_JOSEPH_ADJOINT || kind == YK_BP_SIDDON_ADJOINT) {
        const bool siddon = kind == YK_BP_SIDDON_ADJOINT;
        for (const TransposeRun& r : transpose_runs(siddon, first, count)) {
            transpose(w, siddon, r.form, d_proj + size_t(nu) * nv * (r.first - first), d_volume, r.first, r.count, accumulate);
            accumulate = 1;
        }
    } else if (operator_form(kind)) {
        // a chunk of views (at most 1 GiB) at a time through the paired copy,
        // or all of them without it
        const int chunk = op_chunk(w, count);
        for (int c0 = 0; c0 < count; c0 += chunk > 0 ? chunk : count) {
            OpBpLaunch p = op_launch(kind, d_proj + size_t(nu) * nv * c0, first + c0, chunk > 0 ? std::min(chunk, count - c0) : count);
            p.scale = float(op_scale[first]);
            p.volume = d_volume;
            p.store.mode = c0 > 0 || accumulate ? OpBpStore::kAdd : OpBpStore::kSet;
            p.paired = chunk > 0 ? w.d_paired_views.get() : nullptr;
            launch_fdk_operator_bp(p, s);
        }
    } else {
        fail(YK_ERR_UNSUPPORTED, "unknown back projector");
    }
}

// x += lambda B y / (col + eps), bounded, in the backprojection's own store;
// false when the back model has no such store or takes several launches
bool yk_projector::backproject_update(int kind, const float* d_proj, int first, int count, const OpBpStore& update)
{
    if (!operator_form(kind)) return false;
    yk_projector& w = scratch_owner ? *scratch_owner : *this;
    const int chunk = op_chunk(w, count);
    if (chunk > 0 && chunk < count) return false;
    OpBpLaunch p = op_launch(kind, d_proj, first, count);
    p.store = update;
    p.store.mode = OpBpStore::kUpdate;
    p.paired = chunk > 0 ? w.d_paired_views.get() : nullptr;
    launch_fdk_operator_bp(p, ctx->stream);
    return true;
}

// the backprojections of a view of ones by consecutive units of `counts` views
// from the first on, a volume each in `out`; false when the back model has no
// launch for several units
bool yk_projector::column_weights(int kind, const float* d_ones, const std::vector<int>& counts, bool mask, float* out)
{
    if (!operator_form(kind)) return false;
    yk_projector& w = scratch_owner ? *scratch_owner : *this;
    std::vector<OpBpUnit> units;
    int at = 0;
    for (int k : counts) {
        units.push_back(OpBpUnit{ at, k, float(op_scale[at]), 0 });
        at += k;
    }
    hipStream_t s = ctx->stream;
    if (w.d_op_units.size() < units.size()) w.d_op_units.resize(units.size());
    YK_HIP(hipMemcpyAsync(w.d_op_units.get(), units.data(), units.size() * sizeof(OpBpUnit), hipMemcpyHostToDevice, s));
    OpBpLaunch p = op_launch(kind, d_ones, 0, n_views);
    p.store.mode = mask ? OpBpStore::kWeight : OpBpStore::kSet;
    p.one_view = 1;
    p.paired = op_chunk(w, n_views, true) > 0 ? w.d_paired_views.get() : nullptr;
    // (at most 65535 workgroups along z of a launch)
    const size_t per = std::max<size_t>(1, size_t(60000) / size_t(grid.nz));
    for (size_t k = 0; k < units.size(); k += per) {
        p.units = w.d_op_units.get() + k;
        p.n_units = int(std::min(per, units.size() - k));
        p.volume = out + k * size_t(grid.nx) * grid.ny * grid.nz;
        launch_fdk_operator_bp(p, s);
    }
    YK_HIP(hipStreamSynchronize(s));  // (`units` is host memory)
    return true;
}

// launch of the operator-form backprojection of views [first, first + count)
OpBpLaunch yk_projector::op_launch(int kind, const float* d_proj, int first, int count) const
{
    OpBpLaunch p{};
    p.proj = d_proj;
    p.views = d_opviews.get() + first;
    p.vol = vol;
    p.nu = nu; p.nv = nv; p.count = count;
    p.scale = float(op_scale[first]);
    p.mode = op_mode(kind);
    p.front = std::all_of(op_front.begin() + first, op_front.begin() + first + count, [](char f) { return f != 0; });
    return p;
}

double yk_projector::dot(const float* a, const float* b, size_t n)
{
    hipStream_t s = ctx->stream;
    const int parts = int(std::min<size_t>(1024, std::max<size_t>(1, (n + 255) / 256)));
    launch_dot(a, b, n, d_partials.get(), parts, s);
    std::vector<double> h(parts);
    YK_HIP(hipMemcpyAsync(h.data(), d_partials.get(), parts * sizeof(double), hipMemcpyDeviceToHost, s));
    YK_HIP(hipStreamSynchronize(s));
    double acc = 0.0;
    for (double v : h) acc += v;
    return acc;
}
