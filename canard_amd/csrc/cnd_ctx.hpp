// The context of libcnd (device arrays, tables, sweep shapes) and the
// launch helpers shared by the translation units that launch sweeps.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "../../include/cnd.h"
#include "cnd_dev.hpp"
#include "cnd_scheme.hpp"
#include "cnd_sweepk.hpp"

namespace cnd {
constexpr int kLine = kTile;  // pencils per face/sweep workgroup (one wave)
constexpr int kPts = 256;     // points per pointwise workgroup
// Every block's fields start on a multiple of this many points (2 KiB), so
// that workgroups reading or writing whole tiles of points touch whole
// cache lines of every field; the padding points are never read.
constexpr int64_t kAlignPts = 256;
// stored points from which a context runs independent sweeps side by side
constexpr int64_t kOverlapMinPts = int64_t(4) << 20;
}  // namespace cnd

// Internal header: every translation unit of libcnd works in namespace cnd.
using namespace cnd;

struct OutputState;   // output buffers and writer thread (cnd_output.hip)

// ==== context ===================================================================
// JunctionProgram on the device (one gather and one scatter launch)
struct JuncDev {
    int n = 0;
    int64_t *tgt = nullptr, *src = nullptr;
    int32_t *first = nullptr, *tc = nullptr, *sc = nullptr, *write = nullptr;
    double *scale = nullptr, *tmp = nullptr;
};

// Tiles of a direction that one launch takes (blocks of like pencil length):
// where they start in the direction's list, and their longest pencil.
struct SegClass { int t0, n, S, nmax; };
constexpr int kMaxClasses = 4, kClassTiles = 512;

struct cnd_ctx {
    int ninst = 0, nblk = 0, precision = CND_FP64;
    std::vector<cnd_params> prm;
    std::vector<BlockSpec> spec;
    std::vector<BlkDev> hblk;
    std::vector<Tables> htab;
    std::vector<int64_t> off;
    int64_t NT = 0, FT[3] = {0, 0, 0};
    long long cells = 0;
    int64_t npts = 0;   // stored points (NT, the field stride, also counts the alignment padding)
    hipStream_t st = nullptr;
    // side stream for sweeps that do not depend on each other (eta with
    // zeta gradients, xi with eta fluxes); ev_fork/ev_join order it with st
    hipStream_t st2 = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    bool overlap = true;   // side-by-side sweeps (contexts of >= kOverlapMinPts points; CANARD_OVERLAP)
    BlkDev *dblk = nullptr;
    TabDev *dtab = nullptr;
    InstDev *dinst = nullptr;
    double *dlu = nullptr;
    std::vector<Tile> htiles[3];
    Tile *dtiles[3] = {nullptr, nullptr, nullptr};
    // segmented sweeps: tiles per direction, segments per pencil (rounded to
    // whole waves; 0: the direction uses the tiled sweeps), homogeneous tables
    std::vector<Tile> hstiles[kNumP][3];            // tiles of P pencils, longest pencils first
    std::vector<SegClass> classes[kNumL][kNumP][3];   // launches of segments of L points (seg_classes)
    Tile *dstiles[kNumP][3] = {};
    double *dpk[kNumL] = {};                        // coefficients per L (SegTabs)
    // sweep shape per kind (CND_KIND_*) and direction: index into kShapes
    // or kTiled, with the segments per pencil of the launch (seg_sp)
    int shape[CND_NKIND][3] = {};
    int seg_sp[CND_NKIND][3] = {};
    bool tuned = false, tune_on = true, tiled_only = false;
    bool fuse_update = true;   // last flux sweep writes the RK update (CANARD_FUSE_UPDATE=0: separate)
    int fuse_dir = 0;          // the direction of that sweep, 0 (xi) or 2 (zeta; CANARD_FUSE_DIR=2)
    bool recording = false;    // cnd_record: time averages accumulated in qb
    double *qb = nullptr;
    int lds_max = 65536;   // dynamic LDS per workgroup the device allows
    double tune_ms[CND_NKIND][3] = {};
    std::vector<Tile> hpt;
    Tile *dpt = nullptr;
    // de: right-hand side as three 5-field buffers, one per flux direction
    // (summed in the update); fl: the 15 stored fluxes F[5 d + m], before
    // them a viscous stage's primitives; scratch for metrics, single sweeps and the autotuner otherwise
    double *qa = nullptr, *qo = nullptr, *de = nullptr, *grad = nullptr, *fl = nullptr, *met = nullptr;
    double *ys = nullptr, *xyz = nullptr, *sponge = nullptr, *sp_par = nullptr;
    int nmax[3] = {0, 0, 0};   // longest pencil per direction
    int segs[kNumL][3] = {};   // its segments of L points
    bool part_other[3] = {};   // some block has another block as interface partner along d
    int64_t ys_len = 0;        // doubles in the forward-value scratch
    double *drva[3] = {}, *cmf[3] = {}, *surf[3] = {};
    float *gradf = nullptr;   // mixed precision: the eta and zeta gradients (fields 4 .. 11) in FP32
    JuncDev jn;
    std::vector<char> grid_set;
    bool metrics_ready = false, state_in_qo = false;
    OutputState *out = nullptr;   // created by the first output call
    // the call the stage-by-stage API expects next: 0 a new step (cnd_filter
    // or cnd_step), 1..4 cnd_rk_stage(nk), 5 cnd_end_step
    int next_call = 0;
    bool any_gcbc = false, any_wall = false, any_avg = false, any_sponge = false, any_visc = false;
    bool avg_self = false;    // averaged faces, each between a block and itself
    bool ended = false;       // the step's last averaging has ended the step
    unsigned *tstep_done = nullptr;   // workgroups of k_tstep that are through
    bool any_frame = false;   // some instance's frame accelerates (nsmf = 0)
    // staging of large reads (read_to_host), allocated by the first
    char *stage = nullptr;
    hipEvent_t stage_ev[3] = {};
    bool use_graph = false;
    hipGraphExec_t gexec = nullptr;
    // section timers
    bool prof = false, capturing = false;
    long long launched = 0;    // kernels launched through LAUNCH
    struct Mark { int sec; hipEvent_t a, b; int launches; };
    std::vector<Mark> marks;
    std::vector<hipEvent_t> pool;
    double sec_ms[CND_NSEC] = {};
    long long sec_n[CND_NSEC] = {};
    std::string err;
};

namespace cnd {

// Record message m as the context's (or, without one, the thread's) last
// error and return code.
int fail(cnd_ctx *c, int code, const std::string &m);

#define HIPX(c, call)                                                                               \
    do {                                                                                            \
        hipError_t e_ = (call);                                                                     \
        if (e_ != hipSuccess) return fail((c), CND_EDEVICE, std::string(#call ": ") + hipGetErrorString(e_)); \
    } while (0)


template <class T>
int dalloc(cnd_ctx *c, T **p, size_t n)
{
    HIPX(c, hipMalloc((void **)p, std::max<size_t>(n, 1) * sizeof(T)));
    return CND_OK;
}


inline int check_launch(cnd_ctx *c)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(c, CND_EDEVICE, std::string("kernel launch: ") + hipGetErrorString(e));
    return CND_OK;
}

// Launch helpers ----------------------------------------------------------------
inline dim3 tiles_grid(cnd_ctx *c, int d, int y) { return dim3(unsigned(c->htiles[d].size()), unsigned(y)); }
inline dim3 sweep_grid(cnd_ctx *c, int d, int y) { return dim3(unsigned(xcd_width(int(c->htiles[d].size()))), unsigned(y)); }

// A kernel launch, counted for the section timers.
#define LAUNCH(c, ...)                                                                                     \
    do {                                                                                                   \
        ++(c)->launched;                                                                                   \
        hipLaunchKernelGGL(__VA_ARGS__);                                                                   \
    } while (0)

// Launch a sweep kernel template K<C> with the chunk length of direction d.
#define LAUNCH_SWEEP(K, NV, c, d, y, block, ...)                                                           \
    do {                                                                                                   \
        if ((d) == 0)                                                                                      \
            LAUNCH(c, K<kChunkXi>, sweep_grid(c, d, y), dim3(block),                                       \
                               (sweep_lds_bytes<NV, kChunkXi>()), (c)->st, __VA_ARGS__);                    \
        else                                                                                               \
            LAUNCH(c, K<kChunkEta>, sweep_grid(c, d, y), dim3(block),                                      \
                               (sweep_lds_bytes<NV, kChunkEta>()), (c)->st, __VA_ARGS__);                   \
    } while (0)
inline dim3 pts_grid(cnd_ctx *c) { return dim3(unsigned(c->hpt.size())); }


inline int ntiles(cnd_ctx *c, int d) { return int(c->htiles[d].size()); }
// LDS bytes of a segmented launch (cnd_seg.hpp SegShape).
inline size_t seg_lds_bytes(const ShapeInfo &G, int nv, int sp, int nmax, bool has_part)
{
    const size_t ends = size_t(2) * kSegEndRows * nv * G.P, part = has_part ? ends : 0;
    const size_t ex = size_t(2) * nv * sp * G.P, lu = size_t(5) * G.L * sp, coef = size_t(8) * sp;
    const size_t tile = size_t(nv) * G.P * size_t(nmax | 1) + 2 * kTilePad;   // pencils n | 1 apart (SegShape::pencil_stride)
    if (G.XI) return sizeof(double) * (std::max(tile, lu + ex) + coef + part);
    return sizeof(double) * (std::max(ends, ex) + coef + lu + part);
}

// One segmented launch: shape, tiles, workgroup size and LDS.
struct SegLaunch {
    int shape;
    SegTiles tiles;
    unsigned threads;
    size_t lds;
};

// Eta and zeta sweeps of a kind go in one launch where both have the same
// shape, its LDS serves both, and the lanes the direction with fewer segments
// leaves idle are at most a quarter: a launch of a small block is a chain of
// latencies (10-15 us from 17^3 to 65^3 points), so one launch takes half the
// time of two, and on large blocks it fills the GPU as two streams did.
inline bool eta_zeta_joint(const cnd_ctx *c, int kind)
{
    const int sh = c->shape[kind][1];
    if (sh == kTiled || sh != c->shape[kind][2]) return false;
    const int pi = p_index(kShapes[sh].P), li = l_index(kShapes[sh].L);
    if (c->classes[li][pi][1].size() > 1 || c->classes[li][pi][2].size() > 1) return false;
    const int a = c->segs[li][1], b = c->segs[li][2], m = std::max(a, b);
    // the launch takes the more segments of the one and the partner points of either
    if (seg_lds_bytes(kShapes[sh], 1, std::max(c->seg_sp[kind][1], c->seg_sp[kind][2]), std::max(c->nmax[1], c->nmax[2]),
                      c->part_other[1] || c->part_other[2]) > size_t(c->lds_max))
        return false;
    const int64_t na = int64_t(c->hstiles[pi][1].size()), nb = int64_t(c->hstiles[pi][2].size());
    return 4 * ((m - a) * na + (m - b) * nb) <= m * (na + nb);
}

// Segments per pencil of a workgroup whose pencils have at most S: rounded up
// to whole waves per variable where that fits the shape.
inline int round_sp(const ShapeInfo &G, int S)
{
    const int per_wave = 64 / G.P, up = (S + per_wave - 1) / per_wave * per_wave;
    return up <= G.SPMAX ? up : S;
}

// Launches of nv variables per workgroup for kind along d, one per class of
// pencil lengths; joint: of eta (d = 1) and zeta together.
struct SegLaunches {
    SegLaunch at[kMaxClasses];
    int n = 0;
    const SegLaunch *begin() const { return at; }
    const SegLaunch *end() const { return at + n; }
};
inline SegLaunches seg_launches(const cnd_ctx *c, int kind, int d, int nv, bool joint = false)
{
    const int sh = c->shape[kind][d], pi = p_index(kShapes[sh].P);
    const ShapeInfo &G = kShapes[sh];
    SegLaunches out;
    for (const SegClass &C : c->classes[l_index(G.L)][pi][d]) {
        // (a joint launch has one class per direction)
        const int n2 = joint ? int(c->hstiles[pi][2].size()) : 0;
        const int sp = joint ? std::max(c->seg_sp[kind][1], c->seg_sp[kind][2]) : round_sp(G, C.S);
        const int nmax = joint ? std::max(c->nmax[1], c->nmax[2]) : C.nmax;
        const bool part = c->part_other[d] || (joint && c->part_other[2]);
        out.at[out.n++] = SegLaunch{sh, SegTiles{c->nblk == 1 ? nullptr : c->dstiles[pi][d] + C.t0, C.n + n2, sp, d, C.n},
                                    unsigned(nv * G.P * sp), seg_lds_bytes(G, nv, sp, nmax, part)};
    }
    return out;
}

// Launch the segmented sweep K (a template-id of the shape G, in parentheses)
// as SL (a SegLaunch) says, over xm x its tiles x y workgroups (kernels with xm > 1 split a
// tile's work themselves); the arguments after the common ones follow.
// LAUNCH_SEG*: every launch of SLS (SegLaunches).
#define SEG_CASE(i, K, c, SL, y, ...)                                                                       \
    case i: {                                                                                              \
        using G = Sh##i;                                                                                   \
        LAUNCH(c, K, dim3(unsigned(xcd_width(seg_xm * (SL).tiles.n)), unsigned(y)), dim3((SL).threads),      \
                           (SL).lds, (c)->st, (c)->dblk, (c)->dtab, seg_tabs(c, G::L), (SL).tiles, __VA_ARGS__); \
    } break;
// xi shapes, eta / zeta shapes
#define LAUNCH_SEG_XI(K, c, SLS, xm, y, ...)                                                                \
    for (const SegLaunch &SL : SLS) {                                                                      \
        constexpr int seg_xm = xm;                                                                         \
        switch ((SL).shape) {                                                                               \
            SEG_CASE(0, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(1, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(5, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(7, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(8, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(14, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(15, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(16, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(17, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(18, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(19, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(21, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(22, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(23, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(24, K, c, SL, y, __VA_ARGS__) \
            default: break;                                                                                \
        }                                                                                                  \
    }
#define LAUNCH_SEG_EZ(K, c, SLS, xm, y, ...)                                                                \
    for (const SegLaunch &SL : SLS) {                                                                      \
        constexpr int seg_xm = xm;                                                                         \
        switch ((SL).shape) {                                                                               \
            SEG_CASE(2, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(3, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(4, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(6, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(9, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(10, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(11, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(12, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(13, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(20, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(25, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(26, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(27, K, c, SL, y, __VA_ARGS__) \
            SEG_CASE(28, K, c, SL, y, __VA_ARGS__) \
            default: break;                                                                                \
        }                                                                                                  \
    }
#define LAUNCH_SEG(K, c, SLS, xm, y, ...)                                                                   \
    do {                                                                                                   \
        const SegLaunches sls = SLS;                                                                        \
        if (sls.at[0].tiles.d == 0) { LAUNCH_SEG_XI(K, c, sls, xm, y, __VA_ARGS__) }                         \
        else { LAUNCH_SEG_EZ(K, c, sls, xm, y, __VA_ARGS__) }                                                \
    } while (0)

inline SegTabs seg_tabs(cnd_ctx *c, int L) { return SegTabs{c->dpk[l_index(L)]}; }
inline bool seg_on(const cnd_ctx *c, int kind, int d) { return c->shape[kind][d] != kTiled; }


// Variables per workgroup of a sweep kind along d (flux sweeps run one
// workgroup column per component of the stored fluxes; the eta and zeta
// gradient sweeps, one per stored primitive).
inline int kind_nv(int kind, int d)
{
    return kind == CND_KIND_GRAD && d == 0 ? 4 : 1;
}


// Stages without characteristic faces or sponge fold the update
// into the flux sweep of direction fuse_dir, run after the other two, when
// that sweep is segmented (GCBC needs all three flux derivatives before the
// update; the sponge stays in k_update).
inline bool fuse_possible(const cnd_ctx *c)
{
    return c->fuse_update && !c->any_gcbc && !c->any_sponge;
}


// Sweep launches, one translation unit per sweep kind (cnd_run_*.hip).
// Filter (kind CND_KIND_FILTER) and plain derivative (CND_KIND_FIELD) sweeps
// of nvar fields.
int run_filter_field(cnd_ctx *c, int d, const double *in, double *out, int nvar);
int run_fd_field(cnd_ctx *c, int d, int n45, const double *in, int64_t ivs, double *out, int64_t ovs, int nvar);
// Pencil-end arrays of the flux sweeps.
inline Ends3 ends3(const cnd_ctx *c)
{
    return Ends3{{c->drva[0], c->drva[1], c->drva[2]}, {c->FT[0], c->FT[1], c->FT[2]}};
}

// Viscous stages, in this order.  run_prims: u, v, w, T of the state cur in
// the flux scratch fl, for segmented eta and zeta sweeps.  run_grad: gradient
// sweep along d (kind CND_KIND_GRAD; eta and zeta, xi only where it is the
// tiled one); joint (d = 1): eta and zeta in one launch (eta_zeta_joint).
// run_grad_flux: the xi gradients with the stresses and all fluxes into fl.
inline bool prims_wanted(const cnd_ctx *c)
{
    return c->any_visc && (seg_on(c, CND_KIND_GRAD, 1) || seg_on(c, CND_KIND_GRAD, 2));
}
int run_prims(cnd_ctx *c, const double *cur);
int run_grad(cnd_ctx *c, int d, const double *cur, bool joint = false);
int run_grad_flux(cnd_ctx *c, const double *cur);
// Flux sweep along d into the d-th right-hand-side buffer (kind
// CND_KIND_FLUX) of the stored fluxes, or, where it is a tiled one of an
// inviscid context, of the state cur; joint as for run_grad.
int run_flux(cnd_ctx *c, int d, const double *cur, bool joint = false);
// The directions (bits) whose sweeps take an inviscid stage's stored fluxes.
inline unsigned inv_flux_dirs(const cnd_ctx *c)
{
    unsigned m = 0;
    for (int d = 0; d < 3; ++d) m |= seg_on(c, CND_KIND_FLUX, d) ? 1u << d : 0u;
    return m;
}
// Flux sweep of the stored fluxes along fuse_dir (xi, or zeta) fused with the
// RK update of stage nk, written to qa; the other two directions' buffers
// must be complete.
int run_flux_update(cnd_ctx *c, int nk, double *qa);

// Synchronous copies of device arrays to the caller's host memory, in order
// with st (cnd_read.hip); read_release frees the staging memory (cnd_destroy).
struct HostCopy { void *dst; const void *src; size_t bytes; };
int read_to_host(cnd_ctx *c, const HostCopy *copies, int n);
void read_release(cnd_ctx *c);

// Joins an output write in flight and frees the output buffers (cnd_destroy).
void output_release(cnd_ctx *c);

}  // namespace cnd
