// Internal host-side declarations shared by the C ABI, the plans and the
// kernel launchers of libyk_hip.so.  Nothing here is part of the ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/yk_hip.h"

namespace yk {

// ---------------------------------------------------------------------------
// errors: every failure is a yk::Error carrying a yk_status; the C ABI layer
// converts it to a return code and a thread-local message (no aborts).
// ---------------------------------------------------------------------------
struct Error : std::runtime_error {
    yk_status status;
    Error(yk_status s, const std::string& msg) : std::runtime_error(msg), status(s) {}
};

[[noreturn]] void fail(yk_status status, const std::string& message);
void check_hip(hipError_t err, const char* what);

#define YK_HIP(call) ::yk::check_hip((call), #call)

// ---------------------------------------------------------------------------
// device memory RAII (hipMalloc'd, freed on destruction)
// ---------------------------------------------------------------------------
template <typename T>
class DeviceArray {
public:
    DeviceArray() = default;
    explicit DeviceArray(size_t n) { resize(n); }
    DeviceArray(const DeviceArray&) = delete;
    DeviceArray& operator=(const DeviceArray&) = delete;
    DeviceArray(DeviceArray&& o) noexcept : ptr_(o.ptr_), n_(o.n_) { o.ptr_ = nullptr; o.n_ = 0; }
    DeviceArray& operator=(DeviceArray&& o) noexcept
    {
        if (this != &o) { reset(); ptr_ = o.ptr_; n_ = o.n_; o.ptr_ = nullptr; o.n_ = 0; }
        return *this;
    }
    ~DeviceArray() { reset(); }
    void resize(size_t n)
    {
        if (n == n_) return;
        reset();
        if (n) {
            void* p = nullptr;
            YK_HIP(hipMalloc(&p, n * sizeof(T)));
            ptr_ = static_cast<T*>(p);
            n_ = n;
        }
    }
    void reset()
    {
        if (ptr_) (void)hipFree(ptr_);
        ptr_ = nullptr;
        n_ = 0;
    }
    T* get() const { return ptr_; }
    size_t size() const { return n_; }
    void upload(const T* host, size_t n, hipStream_t s)
    {
        resize(n);
        if (n) YK_HIP(hipMemcpyAsync(ptr_, host, n * sizeof(T), hipMemcpyHostToDevice, s));
    }

private:
    T* ptr_ = nullptr;
    size_t n_ = 0;
};

// pinned host staging buffer (hipHostMalloc'd)
class PinnedBuffer {
public:
    PinnedBuffer() = default;
    PinnedBuffer(const PinnedBuffer&) = delete;
    PinnedBuffer& operator=(const PinnedBuffer&) = delete;
    ~PinnedBuffer() { reset(); }
    void ensure(size_t bytes);
    void reset();
    void* get() const { return ptr_; }

private:
    void* ptr_ = nullptr;
    size_t bytes_ = 0;
};

}  // namespace yk

// ---------------------------------------------------------------------------
// context
// ---------------------------------------------------------------------------
struct yk_ctx {
    int device = 0;
    hipStream_t own_stream = nullptr;
    hipStream_t stream = nullptr;
    bool synchronous = true;
    yk::DeviceArray<double> reduce_scratch;
    yk::PinnedBuffer pinned;
    void finish();  // synchronizes when synchronous, surfaces async errors
    void activate() const;
};

namespace yk {

// ---------------------------------------------------------------------------
// geometry (FP64 host math; float results)
// ---------------------------------------------------------------------------
struct ViewD {
    double src[3], detS[3], detU[3], detV[3];
    double angle;
};

ViewD widen(const yk_view& v);

struct DerivedD {
    double theta, dtheta, fscale, sod, sdd_radial, sdd_plane, off_u, off_v, du, dv;
    double radial[3], normal[3];
    double uu, vv, uv;
};

struct CoeffD {
    double cu[4], cv[4], cd[4], cr[4];
    double wbase;
};

void build_views(const yk_system& system, std::vector<yk_view>& views);
void derive_geometry(const std::vector<yk_view>& views, int nu, int nv, double scan_range,
    std::vector<DerivedD>& out);
void fdk_coefficients(const std::vector<yk_view>& views, const std::vector<DerivedD>& derived,
    std::vector<CoeffD>& out);
void filter_weights(const yk_filter& f, int padded_n, double du, std::vector<float>& out);
// sum of |h[m]| over the padded_n-periodic impulse response h[m] =
// sum_k w[|k|] cos(2 pi k m / padded_n) of the filter weights (FP64): a
// filtered row never exceeds this times the largest |texel| of its input
double filter_response_l1(const std::vector<float>& weights, int padded_n);
void validate_filter(const yk_filter& f);
int padded_n(int nu);
void fft_twiddles(int n, std::vector<float2>& out);
int start_u(int nu, int n, double offset_u_pix);
int main_axis(const yk_view& v, int nu, int nv);
// world point -> detector pixel coordinates: u = (c[0..3].[X,1]) / (c[8..11].[X,1]),
// v = (c[4..7].[X,1]) / (c[8..11].[X,1]); same map as the FDK coefficients
void projection_map(const yk_view& v, double c[12]);

// ---------------------------------------------------------------------------
// device-side records (plain float POD passed to kernels)
// ---------------------------------------------------------------------------
struct alignas(16) BpCoeff {
    float cu[4];   // x y z w
    float cv[4];
    float cd[4];
    float cr[4];
    float wbase;
    float pad[3];
};

struct alignas(16) FilterView {
    float src[4];
    float detS[4];
    float detU[4];
    float detV[4];
    float sdd_radial;
    float wgeom;       // SDD_r / SOD / 2
    int start_u;
    int pad;
};

struct VolumeGeom {
    int nx, ny, nz;
    float vx, vy, vz;
    float ox, oy, oz;  // centre of voxel (0,0,0)
};

VolumeGeom volume_geom(const yk_volume_grid& g);
void validate_volume(const yk_volume_grid& g);

// ---------------------------------------------------------------------------
// kernel launchers (implemented in the .hip translation units)
// ---------------------------------------------------------------------------
struct FilterLaunch {
    const float* proj;          // [count][nv][nu]
    void* out;                  // [count][nv][nu] of `storage`
    float* row_scales;          // [count][nv] (half / bf16)
    const FilterView* views;    // device, `count` records
    const float* parker;        // device [count][nu] Parker weights x range/pi, or null
    const float* weights;       // device, N/2+1
    const float2* twiddles;     // device, N
    int nu, nv, count, n;
    int storage;
    float response_l1;          // filter_response_l1 of `weights` (half / bf16 row scales)
};
void launch_fdk_filter(const FilterLaunch& p, hipStream_t s);
// the cosine (and Parker) weighted projections of p's views into out ([count][nv][nu])
void launch_preweight(const FilterLaunch& p, float* out, hipStream_t s);

struct TileLaunch {
    const double* coeff64;      // device, per view: cu[4] cv[4] cd[4] (12 doubles)
    int n_views;
    VolumeGeom vol;
    int bx, by, bz;             // voxel block
    int nbx, nby, nbz;          // block counts
    int nu, nv;
    short4* tiles;              // [n_blocks][n_views]: u0, v0, width, height (quads)
    uint2* stage;               // [n_blocks][n_views]: staging shape (span reciprocal, chunks, rows)
    int* max_quads;             // device scalars: max width, max height, max staged quads (LDS), bad
};
void launch_bp_tiles(const TileLaunch& p, hipStream_t s);

struct BpLaunch {
    const void* proj;           // [count][nv][nu], storage type
    const unsigned* row_factors; // [count][nv] normalized row factors (half / bf16) or null
    const int* gscale_bits;     // device float bits: max row scale (half / bf16)
    const BpCoeff* coeffs;      // device, `count` records
    const short4* tiles;        // [n_blocks][n_tile_views] with column offset
    const uint2* stage;         // staging shapes, same indexing as tiles
    int tile_view_stride;       // = total views of the plan
    int tile_view_offset;       // first view in the tile table
    float* volume;
    VolumeGeom vol;
    int nu, nv, count;
    int storage;
    int accumulate;
    int kahan;
    int general;                // 0 regular; 1 / 2 u varies along z (tilted detector):
                                // a reciprocal per sample / Newton steps (fdk.cpp general_mode)
    int nbx, nby, nbz;
    int bz;                     // z slices per workgroup (32, 16 or 8)
    int lds_quads;              // LDS capacity in quads
    int parts;                  // parts of part_views views each, in workgroups of their own
    int part_views;
    float* part_volumes;        // `parts` volumes when parts > 1
};
void launch_fdk_bp(const BpLaunch& p, hipStream_t s);
// BpLaunch::storage of half texels already normalized by launch_normalize_rows
constexpr int kBpHalfNormalized = 16;
// rows x nu half / bfloat16 texels times their normalized row factors -> half
void launch_normalize_rows(const void* in, const unsigned* factors, int storage, int rows, int nu, void* out,
    hipStream_t s);
// global maximum row scale into *gbits, then per row the factor scale / max
// (packed half pair for half storage, float bits for bfloat16)
void launch_row_factors(const float* scales, int n, int storage, int* gbits, unsigned* factors,
    hipStream_t s);
int bp_block_z(int general, int storage, int kahan);
// bytes of one LDS quad of the backprojection: 16 (float) for float storage
// and for every storage of a general-geometry plan, 8 (half) otherwise
size_t bp_quad_bytes(int storage, int general);
// progress report of the iterative callers: waits for the stream's work, then
// calls cb(user, completed, total) on this thread; no-op without a callback
void report_progress(yk_progress_fn cb, void* user, int completed, int total, hipStream_t s);
// Fixed per-GPU scratch of the allocation-free backprojection: a header of
// kNoAllocHeader words (word 0: global row-scale bits) and room for
// kNoAllocRowFactors row factors (views x detector rows of one call).
constexpr size_t kNoAllocHeader = 64;
constexpr size_t kNoAllocRowFactors = size_t(YK_NOALLOC_MAX_ROWS);
// device address of that array on `device` (must be the current device),
// looked up with hipGetSymbolAddress on the first call for the device
unsigned* bp_noalloc_scratch(int device);

struct ProjViewDev {
    float src[4];               // voxel-normalized, volume-centred
    float detS[4];
    float detU[4];
    float detV[4];
    int axis;                   // 0 X, 1 Y, 2 Z
    int pad[3];
};

struct SiddonViewDev {
    float src[4];               // world
    float detS[4];
    float detU[4];
    float detV[4];
    int plane[4];               // per axis, the plane between cells that the source lies on, or -1 (projector.cpp)
    float on_plane[4];          // src, moved onto that plane as the gathers form it
};

struct JosephLaunch {
    const float* volume;        // [z][y][x]
    const float* volume_t;      // [z][x][y] copy, for axis-X views (may be null)
    float* proj;                // [count][nv][nu]
    const ProjViewDev* views;   // device, `count`
    VolumeGeom vol;
    int nu, nv, count;
    int accumulate;
};
void launch_joseph_fp(const JosephLaunch& p, hipStream_t s);
void launch_joseph_ones(const JosephLaunch& p, hipStream_t s);  // of a volume of ones (volume unused)
void launch_transpose_xy(const float* in, float* out, int nx, int ny, int nz, hipStream_t s);

// what becomes of a projected value a: proj =, proj +=, or the algebraic
// solvers' residual, proj = row > eps ? (b - a) / row : 0 or proj = (b - a) row
struct FpStore {
    enum Mode { kSet, kAdd, kResidualDivide, kResidualMultiply };
    int mode;
    float eps;
    const float* b;             // views b_view floats apart
    const float* row;           // as proj
    size_t b_view;
};

// Joseph projection from volume copies
struct JosephSepFpLaunch {
    const float* vol_zx;        // copy for X-main views (may be null if none)
    const float* vol_zy;        // copy for Y-main views (may be null if none)
    float* proj;                // [count][nv][nu]
    const ProjViewDev* views;   // device, `count`
    VolumeGeom vol;
    int nu, nv, count;
    FpStore store;
};
// separable views, from Z-fastest copies (launch_joseph_column_copy) of
// joseph_column_size floats: [slice][row][z] of a [z][y][x] volume, slices along
// the main axis (x for x_main, else y), rows along the other of x and y, two
// zero planes before and after each minor axis
void launch_joseph_fp_column(const JosephSepFpLaunch& p, hipStream_t s);
void launch_joseph_column_copy(const float* in, float* out, int nx, int ny, int nz, bool x_main, hipStream_t s);
size_t joseph_column_size(int nx, int ny, int nz, bool x_main);
bool joseph_column_fits(const VolumeGeom& g);
// X- or Y-main views of any orientation, from paired slab copies
// (launch_joseph_pair_copy) of joseph_pair_size floats: float2 entries (value
// at z row r, value at row r + 1), columns along the other of x and y, two
// zero planes around both minor axes.  A copy raises *flag (null: unused) for
// values that launch_siddon_fp_slab cannot take.
void launch_joseph_fp_slab(const JosephSepFpLaunch& p, hipStream_t s);
void launch_joseph_pair_copy(const float* in, float* out, int nx, int ny, int nz, bool x_main, hipStream_t s,
    int* flag = nullptr);
void launch_clear_flag(int* flag, hipStream_t s);
size_t joseph_pair_size(int nx, int ny, int nz, bool x_main);

struct JosephAdjointLaunch {
    const float* proj;          // [count][nv][nu]
    float* volume;              // [z][y][x]
    const ProjViewDev* views;   // device, `count`
    const float* coeff32;       // device, per view cu[4] cv[4] cd[4] (world projective map)
    float4* ray_ab;             // scratch [count][nv][nu]: a1, b1, a2, b2 of every ray
    float* ray_len;             // scratch [count][nv][nu]: L (0: ray skipped)
    VolumeGeom vol;
    int nu, nv, count;
    int accumulate;
};
void launch_joseph_adjoint(const JosephAdjointLaunch& p, hipStream_t s);

// per-view record of the gather transposes (kernels_gather.hip): the map that
// bounds the candidates of either model and, for Joseph, source and pixel
// offsets in volume-centred voxel units, component 0 the main axis, 1 the
// other of x and y, 2 z; pixel minus source is d / e1 / e2 = [0] + u [1] +
// v [2] on components 0 / 1 / 2, times `scale`, a power of two that brings |d|
// into [0, 1] over the detector
struct GatherViewDev {
    double src[3];
    double d[3], e1[3], e2[3];
    float mu[4], mv[4], md[4];  // projective map of voxel indices [x, y, z, 1]: u = mu / md, v = mv / md
    float scale;
    int axis;                   // 0 X, 1 Y
};

// (flat: separable views whose row steps have no z component; ends: rays may end
// inside the volume)
enum GatherModel { kGatherJoseph, kGatherSiddon, kGatherSiddonFlat, kGatherSiddonFlatEnds };
struct GatherLaunch {
    const float* proj;          // [count][nv][nu]
    float* volume;              // [z][y][x]
    const ProjViewDev* views;   // device, `count` (Joseph)
    const SiddonViewDev* sviews; // device, `count` (Siddon)
    const GatherViewDev* gviews; // device, `count`
    float* q;                   // scratch [count][nv + kGatherPadRows][pitch] floats or float triples (kGatherSiddon)
    float2* ru;                 // scratch [count][pitch] (kGatherSiddonFlat)
    float* rv;                  // scratch [count][nv + kGatherPadRows] (kGatherSiddonFlat)
    int* flag;                  // scratch word
    VolumeGeom vol;
    int nu, nv, pitch, count;
    int model;
    int accumulate;
};
void launch_gather_transpose(const GatherLaunch& p, hipStream_t s);
// zero columns closing each row, and zero rows closing each view, of the
// gather transposes' table (a chunk of candidates may run past the last pixel)
constexpr int kGatherPad = 4;
constexpr int kGatherPadRows = 3;
constexpr int kGatherRun = 8;  // voxels along z of a lane

// Joseph transpose of separable views by detector columns (kernels_column.hip)
struct ColumnTransposeLaunch {
    const float* proj;          // [count][nv][nu]
    float* volume;              // [z][y][x]
    const ProjViewDev* views;   // device, `count`
    const GatherViewDev* gviews; // device, `count`
    float* q;                   // scratch [count][nu][pitch], pitch = nv + 2 kColumnPad
    float* part_x;              // scratch [x][y][z] (null: no X-main view)
    float* part_y;              // scratch [y][x][z] (null: no Y-main view)
    int* flag;                  // scratch word
    VolumeGeom vol;
    int nu, nv, pitch, count;
    int accumulate;
};
void launch_joseph_column_transpose(const ColumnTransposeLaunch& p, hipStream_t s);
constexpr int kColumnPad = 8;      // zeros on either side of a table's column
constexpr int kColumnSlices = 4;   // consecutive slices of a workgroup, a wave each
constexpr int kColumnGroups = 4;   // 64-voxel groups along z of a wave, at most

struct SiddonLaunch {
    const float* volume;
    float* proj;
    const SiddonViewDev* views;
    VolumeGeom vol;
    int nu, nv, count;
    int accumulate;
};
void launch_siddon_fp(const SiddonLaunch& p, hipStream_t s);
void launch_siddon_ones(const SiddonLaunch& p, hipStream_t s);  // of a volume of ones (volume unused)

// Siddon projection over the paired slab copies of the volume
// (launch_joseph_pair_copy).  The main axis is chosen per ray: a copy may be null
// if no ray of the call has its axis.
struct SiddonSlabFpLaunch {
    const float* volume;        // [z][y][x]
    const float* vol_x;         // paired slab copy, X-main
    const float* vol_y;         // paired slab copy, Y-main
    const int* flag;            // raised by the copies: the volume holds values only the walk can carry
    float* proj;                // [count][nv][nu]
    const SiddonViewDev* views; // device, `count`
    VolumeGeom vol;
    int nu, nv, count;
    int accumulate;
};
void launch_siddon_fp_slab(const SiddonSlabFpLaunch& p, hipStream_t s);

struct SiddonAdjointLaunch {
    const float* proj;
    float* volume;
    const SiddonViewDev* views;
    const float* coeff32;  // the projective map in float, 12 per view
    VolumeGeom vol;
    int nu, nv, count;
    int accumulate;
};
void launch_siddon_adjoint(const SiddonAdjointLaunch& p, hipStream_t s);

// Transposes of untilted views by scattering (kernels_scatter.hip); the ray table
// arrays are scratch of `count` views, columns closed by kScatterPad zero entries
constexpr int kScatterPad = 8;
struct JosephScatterLaunch {
    const float* proj;          // [count][nv][nu]
    float* volume;              // [z][y][x]
    const ProjViewDev* views;   // device, `count`
    const float* coeff32;       // device, per view cu[4] cv[4] cd[4] (world projective map)
    float2* ab1;                // scratch [count][nu]
    float2* ab2;                // scratch [count][nu][nv + kScatterPad]
    float* pl;                  // scratch [count][nu][nv + kScatterPad]
    VolumeGeom vol;
    int nu, nv, count;
    int accumulate;
};
void launch_joseph_scatter(const JosephScatterLaunch& p, hipStream_t s);
struct SiddonScatterLaunch {
    const float* proj;          // [count][nv][nu]
    float* volume;              // [z][y][x]
    const SiddonViewDev* views; // device, `count`
    const float* coeff32;       // device, per view cu[4] cv[4] cd[4] (world projective map)
    float2* col_xy;             // scratch [count][nu]
    float2* ray_wz;             // scratch [count][nu][nv + kScatterPad]
    VolumeGeom vol;
    int nu, nv, count;
    int accumulate;
};
void launch_siddon_scatter(const SiddonScatterLaunch& p, hipStream_t s);

// per-view record of the operator-form FDK backprojections (world units)
struct OpBpViewDev {
    float cu[4], cv[4], cd[4];  // projective map u = Cu.[X,1] / Cd.[X,1], v likewise
    float cc[4];                // FDK weight denominator (-src / SOD, SOD)
    float src[4];
    float l2[6];                // |detS + u detU + v detV - src|^2: 1, u, v, uu, uv, vv
    float wbase;                // SOD^2 dtheta fscale
    float inv_sdd_plane;
};

// views [first, first + count) of a launch's, backprojected into a volume of their own
struct OpBpUnit {
    int first, count;
    float scale;
    int pad;
};

// what becomes of a backprojected value
struct OpBpStore {
    enum Mode { kSet, kAdd, kWeight, kUpdate };
    int mode;                   // volume =, volume +=, volume = (value > 0 ? value : 1e30), x += lambda value / (col + eps)
    float* x;                   // (kUpdate) then bounded
    const float* col;
    float lambda, eps;
    int use_min, use_max;
    float lo, hi;
};

struct OpBpLaunch {
    const float* proj;          // [count][nv][nu], unfiltered
    float* volume;              // [z][y][x]
    const OpBpViewDev* views;   // device, `count`
    VolumeGeom vol;
    int nu, nv, count;
    float scale;                // vx vy vz / (du dv) of the first view (matched weight)
    int mode;                   // 0 FDK weight, 1 pseudo-matched, 2 voxel-driven Joseph
    OpBpStore store;
    const OpBpUnit* units;      // device, n_units, volume [unit][z][y][x]; null: one unit of `count` views
    int n_units;
    int one_view;               // every view has the pixels of proj's first
    int front;                  // every voxel lies before every source, with regular weights (projector.cpp)
    float* paired;              // scratch of count x paired_view_floats: sample a paired copy (null: the views)
};
size_t paired_view_floats(int nu, int nv);
void launch_fdk_operator_bp(const OpBpLaunch& p, hipStream_t s);

// vector helpers
void launch_dot(const float* a, const float* b, size_t n, double* partials, int n_partials,
    hipStream_t s);
void launch_axpy(float* y, const float* x, float a, size_t n, hipStream_t s);        // y += a x
void launch_xpby(float* y, const float* x, float b, size_t n, hipStream_t s);        // y = x + b y
void launch_scale_copy(float* y, const float* x, float a, size_t n, hipStream_t s);  // y = a x
void launch_fill(float* y, float v, size_t n, hipStream_t s);
// algebraic steps: mode 0 res = row > eps ? (b - res) / row : 0, mode 1 res = (b - res) row,
// over `count` views of view_n values; consecutive views of b lie b_stride views apart
void algebraic_residual(float* res, const float* b, const float* row, float eps, int mode, size_t view_n, int count,
    int b_stride, hipStream_t s);
// x += lambda bp / (col + eps), then optional bounds
void algebraic_update(float* x, const float* bp, const float* col, float lambda, float eps, int use_min,
    float lo, int use_max, float hi, size_t n, hipStream_t s);
void launch_bounds_clamp(float* x, int use_min, float lo, int use_max, float hi, size_t n, hipStream_t s);
// x <= threshold -> 1e30, then optionally x = 1 / x
void weight_prepare(float* x, float threshold, int reciprocal, size_t n, hipStream_t s);
// smoothed TV value partials and gradient; dims 3 (volume) or 2 (each z slice alone)
// (16 workgroups a CU: with four, and three 64-bit divisions a voxel for its
// place, an OS-SART sweep with three steps on 1.6 million voxels took 1.304 ms
// instead of 1.285)
// Smaller volumes have a quarter, which the value's sum copies to the host:
// 48^3 29.3 -> 25.8 us a call, 96^3 34.2 -> 31.6.
constexpr int kTvPartials = 4096;
inline int tv_partials(const VolumeGeom& g) { return double(g.nx) * g.ny * g.nz < 1e6 ? kTvPartials / 4 : kTvPartials; }
void launch_tv_gradient(const float* x, float* grad, double* partials, int n_partials,
    const VolumeGeom& g, float eps, hipStream_t s, int dims = 3);
void launch_phantom(const float* ellipsoids, int n, const VolumeGeom& g, int clamp,
    float* out, hipStream_t s);

}  // namespace yk
