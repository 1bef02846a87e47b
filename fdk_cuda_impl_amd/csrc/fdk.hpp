// FDK plan and projection-operator plan (library-owned handles of the C ABI).
#pragma once

#include <atomic>
#include <memory>
#include <string>
#include <vector>

#include "yk_internal.hpp"

struct yk_fdk {
    yk_fdk(yk_ctx* ctx, const yk_fdk_desc& desc, const yk_view* views, int n_views, int nu,
        int nv, const yk_volume_grid& grid);

    void filter(const float* d_proj, int first, int count, void* d_out, int storage, float* d_scales,
        float* d_preweighted = nullptr);
    void backproject(const void* d_filtered, int storage, const float* d_scales, int first, int count,
        float* d_volume, int accumulate);
    // backproject() with no device allocation (scratch in the fixed per-GPU array)
    void backproject_noalloc(const void* d_filtered, int storage, const float* d_scales, int first, int count,
        float* d_volume, int accumulate);
    void execute(const float* projection, int ploc, size_t pcap, int offset, int count, float* volume,
        int vloc, size_t vcap, int clear_output);

    yk_ctx* ctx;
    yk_fdk_desc desc;
    int nu, nv, n_views;
    yk_volume_grid grid;
    yk::VolumeGeom vol{};
    double scan_range = 0.0;
    bool parker = false;
    bool general = false;
    int geo_mode = 0;              // 0 regular, 1 tilted (reciprocal per sample), 2 tilted (Newton steps)
    std::vector<yk_view> views;
    std::vector<yk::DerivedD> derived;
    std::vector<yk::CoeffD> coeffs;
    std::vector<float> weights;
    int n_pad = 0;
    float response_l1 = 0.f;       // filter_response_l1 of weights

    yk::DeviceArray<float> d_weights;
    yk::DeviceArray<float2> d_twiddles;
    yk::DeviceArray<yk::FilterView> d_fviews;
    yk::DeviceArray<yk::BpCoeff> d_coeffs;
    yk::DeviceArray<double> d_c64;
    yk::DeviceArray<float> d_parker;
    yk::DeviceArray<short4> d_tiles;
    yk::DeviceArray<uint2> d_stage;
    yk::DeviceArray<int> d_maxes;      // [0..3] footprint maxima, [4] global row-scale bits
    yk::DeviceArray<unsigned> d_rowfac; // normalized row factors of the views being backprojected
    yk::DeviceArray<unsigned short> d_norm_ws; // half texels times their row factors (half / bf16 storage)
    int nbx = 0, nby = 0, nbz = 0, bz = 0;
    int lds_quads = 0;

    int batch = 0;
    yk::DeviceArray<float> d_proj_ws;     // host projections: two staged chunks
    // Host buffers move through two library-owned pinned slots: the host
    // copies a chunk into a slot with several threads while the copy stream
    // moves the other slot to the device and the plan's stream filters and
    // backprojects the chunk before (stage_chunk_views()).
    yk::PinnedBuffer pinned[2];
    hipStream_t copy_stream = nullptr;   // default priority
    hipEvent_t ev_pinned[2] = {};        // slot's last transfer done (host may reuse it)
    hipEvent_t ev_consumed[2] = {};      // filter of the slot's device chunk done
    bool pinned_used[2] = {};
    bool consumed_used[2] = {};
    int stage_chunk_views() const;
    void ensure_staging(size_t slot_bytes);
    void upload_host(float* d_dst, const float* host, size_t bytes);
    void download_host(float* host, const float* d_src, size_t bytes);
    ~yk_fdk();
    yk::DeviceArray<unsigned char> d_filtered_ws;
    yk::DeviceArray<float> d_scales_ws;
    yk::DeviceArray<float> d_volume_ws;
    int received = 0;

    // calibrated-geometry report (diagnostics.cpp) and the last chunk's stages
    yk_geometry_diagnostics diagnostics{};
    bool capture_stages = false;
    yk::DeviceArray<float> d_preweighted_ws;
    yk_fdk_stage last_stage{};

private:
    void build_tiles();
    int part_count(int count) const;
    void split_views(yk::BpLaunch& p) const;
    yk::DeviceArray<float> d_parts;    // the parts' volumes of a small volume's backprojection
};

struct yk_projector;

// What the algebraic solvers keep with their projector between calls: work
// arrays, and operators made from its views (their contents hold nothing from
// one call for the next).  Arrays beyond kKeep bytes in all are given back
// when the call ends; the rest with the projector.
struct SolverScratch {
    static constexpr size_t kKeep = size_t(1) << 30;
    yk::DeviceArray<float> arrays[8];
    std::unique_ptr<yk_projector> subset_op;  // the views in the order of subset_op_units interleaved subsets
    int subset_op_units = 0;
    std::unique_ptr<yk_projector> coarse;     // the TIGRE row weights' support volume
    // array k with room for n floats; another call's array of any size is kept
    // if it has
    float* array(int k, size_t n);
    ~SolverScratch();
    std::atomic<bool> busy{ false };
};

// One solver call: takes the projector's scratch, or scratch of its own where
// another call (a progress callback's, another thread's) holds that; its queued
// work is done and the large arrays are freed when it ends, by return or by error
struct SolverCall {
    SolverScratch own;
    SolverScratch& ws;
    hipStream_t stream;
    SolverCall(SolverScratch& kept, hipStream_t s) : ws(kept.busy.exchange(true) ? own : kept), stream(s) {}
    SolverCall(const SolverCall&) = delete;
    SolverCall& operator=(const SolverCall&) = delete;
    ~SolverCall();
};

struct yk_projector {
    // `segments`: counts of consecutive views that are view sequences of their
    // own for the operator-form backprojections (null: all views are one)
    yk_projector(yk_ctx* ctx, const yk_view* views, int n_views, int nu, int nv,
        const yk_volume_grid& grid, float scan_range, const std::vector<int>* segments = nullptr);

    // `residual`: the store to make of the values where the kernel has it; false
    // when they are stored as they are
    bool project(int kind, const float* d_volume, float* d_proj, int first, int count, int accumulate,
        const yk::FpStore* residual = nullptr);
    void project_ones(int kind, float* d_proj, int first, int count);  // of a volume of ones
    void backproject(int kind, const float* d_proj, float* d_volume, int first, int count, int accumulate);
    bool backproject_update(int kind, const float* d_proj, int first, int count, const yk::OpBpStore& update);
    bool column_weights(int kind, const float* d_ones, const std::vector<int>& counts, bool mask, float* out);
    yk::OpBpLaunch op_launch(int kind, const float* d_proj, int first, int count) const;
    bool column_transpose(yk_projector& w, const float* d_proj, float* d_volume, int first, int count, int accumulate);
    double dot(const float* a, const float* b, size_t n);
    bool siddon_copies(yk_projector& w, const float* d_volume, bool any_x, bool any_y);
    int op_chunk(yk_projector& w, int count, bool one_view = false) const;
    bool gather_transpose(yk_projector& w, int model, const float* d_proj, float* d_volume, int first, int count, int accumulate);
    enum TransposeForm { kUntilted, kGeneral, kScatter, kSearch };
    struct TransposeRun {
        TransposeForm form;
        int first, count;
    };
    std::vector<TransposeRun> transpose_runs(bool siddon, int first, int count) const;
    bool scatter_transpose(yk_projector& w, bool siddon, const float* d_proj, float* d_volume, int first, int count,
        int accumulate);
    void transpose(yk_projector& w, bool siddon, TransposeForm form, const float* d_proj, float* d_volume, int first, int count,
        int accumulate);

    yk_ctx* ctx;
    int nu, nv, n_views;
    yk_volume_grid grid;
    yk::VolumeGeom vol{};
    double scan_range;
    std::vector<yk_view> views;
    bool any_x_axis = false;
    yk::DeviceArray<yk::ProjViewDev> d_jviews;
    yk::DeviceArray<yk::SiddonViewDev> d_sviews;
    yk::DeviceArray<float> d_c32;      // the projective map in float (transpose candidates)
    yk::DeviceArray<float4> d_ray_ab;  // Joseph transpose ray table, one view chunk
    yk::DeviceArray<float> d_ray_len;
    std::vector<char> separable;       // per view: main axis X/Y and detV along Z only
    // projector whose scratch arrays (volume copies, ray tables) this one uses;
    // null: its own.  Operators of one volume grid that run one after another
    // on one stream can share them.
    yk_projector* scratch_owner = nullptr;
    // Scratch only grows: paths of different layouts share an array, and a
    // reallocation would synchronize.  Once a call has been captured into a graph an
    // array that has to grow is kept beside its successor until the projector goes:
    // the graph's replays go on using it.
    template <typename T>
    void grow(yk::DeviceArray<T>& a, size_t n)
    {
        if (a.size() >= n) return;
        if (captured && a.size()) retired.push_back(std::make_shared<yk::DeviceArray<T>>(std::move(a)));
        a.resize(n);
    }
    void note_capture();               // sets the two flags for a call about to be made
    bool capturing = false, captured = false;
    std::vector<std::shared_ptr<void>> retired;
    yk::DeviceArray<float> d_vol_t;
    yk::DeviceArray<float> d_vol_zx;   // paired volume copies of the Joseph and Siddon projections
    yk::DeviceArray<float> d_vol_zy;
    std::vector<char> siddon_flat;     // per view: siddon_flat_gather covers it
    std::vector<char> siddon_ends;     // per view: the detector may end rays inside the volume
    std::vector<char> joseph_column;   // per view: the column transpose covers it
    yk::DeviceArray<float> d_column_x, d_column_y;  // its volumes of the X- and Y-main views
    std::vector<char> joseph_gather, siddon_gather;  // per view: the gather transposes cover it
    std::vector<char> near_source;     // per view: a voxel lies within their margin of the source plane, or behind it
    yk::DeviceArray<yk::GatherViewDev> d_gather;
    yk::DeviceArray<float> d_scatter;  // ray table of the scatter transposes, one view chunk
    yk::DeviceArray<float> d_gather_q; // ray values of the gather transposes, one view chunk
    yk::DeviceArray<float> d_paired_views;  // paired views of the operator-form backprojections, one chunk
    yk::DeviceArray<int> d_flag;       // one word: a copy or table holds values of an extreme size
    std::vector<char> siddon_axes;     // per view: bit 0, 1: some ray may have the main axis X, Y
    yk::DeviceArray<double> d_partials;
    yk::DeviceArray<yk::OpBpViewDev> d_opviews;  // operator-form FDK backprojection records
    yk::DeviceArray<yk::OpBpUnit> d_op_units;  // units of a column_weights launch
    std::vector<char> op_front;        // per view: no voxel needs the operator backprojections' sample tests
    std::vector<double> op_scale;      // per first view: vx vy vz / (du dv)
    SolverScratch solver;
};

// unified SIRT / SART / OS-SART (algebraic.cpp); throws through fail()
void run_algebraic(yk_projector* p, const yk_algebraic_desc& d, const float* d_b, float* d_x,
    yk_iterative_stats* stats);
// CGLS, robust-restart and ASTRA strategies (cgls.cpp); throws through fail()
void run_cgls(yk_projector* p, const yk_cgls_desc& d, const float* d_b, float* d_x, yk_iterative_stats* stats,
    double* residual_norms);

// calibrated-geometry diagnostics (diagnostics.cpp); throws INVALID_GEOMETRY
// for geometry FDK cannot use
void geometry_diagnostics(const std::vector<yk_view>& views, const std::vector<yk::DerivedD>& derived,
    yk_geometry_diagnostics& out);
// raw dumps (diagnostics.cpp)
std::string dump_name_a(const char* prefix, int a, const char* ext);
yk_dump* dump_create(const char* dir, int enabled);
void dump_destroy(yk_dump* d);
void dump_set_enabled(yk_dump* d, int on);
void dump_device_f32(yk_dump* d, const std::string& name, const float* src, size_t count, hipStream_t s);
void dump_text(yk_dump* d, const std::string& name, const char* text);
